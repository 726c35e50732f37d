// The module-level helpers of sandmuon/optimizer.py, in the dtype of their
// inputs (FP32 or FP64, as the reference computes them):
//   diagonal_inverse_sqrt (:19-24) and rank1_inverse_sqrt (:27-35)
//                         -> smx_inverse_sqrt (one block per vector);
//   rank1_whiten (:38-45) and rank1_mapback (:48-60) -> smx_rank1_apply;
//   _graft_direction (:63-66) -> smx_graft (FP32, as the reference).
// The optimizer's own step uses the fused one-sided kernels of matrix.hip
// and the batched finish of stats.hip; these entry points serve direct
// calls of the helpers.
//
// rank1_apply, with t_j = sum_i lz_i V_ij and u_i = sum_j V_ij rz_j (sums in
// FP64, rounded to T):
//   whiten  (order 0): V0 = (X li) ri;  V1 = V0 + (lc lz_i) t_j;
//                      out = V1 + (rc u_i) rz_j
//   mapback (order 1): V1 = X + (lc lz_i) t_j;  V2 = V1 + (rc u_i) rz_j;
//                      out = (V2 li) ri
// in two launches: column sums (a block per 32 columns, 32 row groups),
// then the rows (one or four waves each: their sums, then their output).
#include "common.h"

#include <algorithm>
#include <cfloat>
#include <cmath>

namespace smx {

template <typename T>
struct Rank1Args {
  const T *x;
  T *out;
  int64_t rows, cols;
  const T *li, *lz, *lc;  // [batch or 1][rows], [batch or 1][rows], [batch or 1]
  const T *ri, *rz, *rc;  // [batch or 1][cols], [batch or 1][cols], [batch or 1]
  double *t;              // [batch][cols] column sums lz^T V
  int32_t order;
  int64_t lb, rb;         // 1, or 0 where one left (right) factor serves the whole batch
};

// The first-stage value V0 (whiten) or X (mapback) of element (i, j).
template <typename T>
__device__ __forceinline__ T r1_v0(const Rank1Args<T> &a, int64_t b, int64_t i, int64_t j) {
  const T x = a.x[(b * a.rows + i) * a.cols + j];
  return a.order == 0 ? (x * a.li[a.lb * b * a.rows + i]) * a.ri[a.rb * b * a.cols + j] : x;
}

// t[b][j] = sum_i lz_i V0_ij: a block takes kColTile columns, its kColRows
// row groups every kColRows-th row each, kColUnroll loads in flight per
// thread, then the groups in order through LDS.  Bound by latency at helper
// sizes: a thread's chain is rows / kColRows terms (one chain of all rows
// per column: 173 us for [4, 640, 1280], this one 11).
// grid (ceil(cols / kColTile), batch), block kColTile x kColRows.
constexpr int kColTile = 32, kColRows = 32, kColUnroll = 4;
template <typename T>
__global__ void __launch_bounds__(kColTile * kColRows) rank1_colsum_kernel(Rank1Args<T> a) {
  __shared__ double part[kColRows][kColTile];
  const int64_t b = blockIdx.y;
  const int lane = threadIdx.x % kColTile, grp = threadIdx.x / kColTile;
  const int64_t j = static_cast<int64_t>(blockIdx.x) * kColTile + lane;
  double s = 0.0;
  if (j < a.cols)
    for (int64_t i0 = grp; i0 < a.rows; i0 += kColRows * kColUnroll) {
      double lz[kColUnroll], v[kColUnroll];
#pragma unroll
      for (int u = 0; u < kColUnroll; ++u) {
        const int64_t i = i0 + kColRows * u;
        const bool in = i < a.rows;
        lz[u] = in ? static_cast<double>(a.lz[a.lb * b * a.rows + i]) : 0.0;
        v[u] = in ? static_cast<double>(r1_v0(a, b, i, j)) : 0.0;
      }
#pragma unroll
      for (int u = 0; u < kColUnroll; ++u)
        if (i0 + kColRows * u < a.rows) s += lz[u] * v[u];
    }
  part[grp][lane] = s;
  __syncthreads();
  if (grp == 0 && j < a.cols) {
    for (int g = 1; g < kColRows; ++g) s += part[g][lane];
    a.t[b * a.cols + j] = s;
  }
}

// A row by kW waves: u_i = sum_j V1_ij rz_j (FP64), then the row's output,
// from registers where the row is one round of kRowUnroll columns per lane
// and else from a second read.  Bound by latency at helper sizes: four waves
// per row give a CU 40 waves for [4, 640, 1280] (11 us), where one wave per
// row left it at 10 with five rounds in series (22 us).
// grid (ceil(rows kW / 4), batch), block 256.
constexpr int kRowUnroll = 8;
template <typename T, int kW>
__global__ void __launch_bounds__(256) rank1_row_kernel(Rank1Args<T> a) {
  __shared__ double part[4];
  constexpr int kLanes = 64 * kW, kRound = kLanes * kRowUnroll;
  const int64_t b = blockIdx.y;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * (4 / kW) + threadIdx.x / kLanes;
  if (i >= a.rows) return;  // uniform over the row's waves
  const int lane = threadIdx.x % kLanes;
  const T li = a.li[a.lb * b * a.rows + i];
  const T cl = a.lc[a.lb * b] * a.lz[a.lb * b * a.rows + i];
  const T *x = a.x + (b * a.rows + i) * a.cols;
  T *out = a.out + (b * a.rows + i) * a.cols;
  const T *ri = a.ri + a.rb * b * a.cols, *rz = a.rz + a.rb * b * a.cols;
  const double *t = a.t + b * a.cols;
  const bool whiten = a.order == 0;
  T v[kRowUnroll], r[kRowUnroll], z[kRowUnroll];  // V1, ri and rz of the lane's columns of one round
  auto load = [&](int64_t j0) {
    T c[kRowUnroll];
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) {
      const int64_t j = j0 + kLanes * u;
      const bool in = j < a.cols;
      v[u] = in ? x[j] : static_cast<T>(0);
      r[u] = in ? ri[j] : static_cast<T>(0);
      z[u] = in ? rz[j] : static_cast<T>(0);
      c[u] = in ? static_cast<T>(t[j]) : static_cast<T>(0);
    }
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) v[u] = (whiten ? (v[u] * li) * r[u] : v[u]) + cl * c[u];
  };
  double s = 0.0;
  for (int64_t j0 = lane; j0 < a.cols; j0 += kRound) {
    load(j0);
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u)
      if (j0 + kLanes * u < a.cols) s += static_cast<double>(v[u]) * static_cast<double>(z[u]);
  }
  s = kW == 1 ? wave_sum(s) : block_sum(s, part);
  const T cu = a.rc[a.rb * b] * static_cast<T>(s);
  for (int64_t j0 = lane; j0 < a.cols; j0 += kRound) {
    if (a.cols > kRound) load(j0);
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) {
      const int64_t j = j0 + kLanes * u;
      if (j >= a.cols) continue;
      T w = v[u] + cu * z[u];
      if (!whiten) w = (w * li) * r[u];
      out[j] = w;
    }
  }
}

template <typename T>
static int launch_rank1(const Rank1Args<T> &a, int64_t batch, hipStream_t st) {
  const unsigned nb = static_cast<unsigned>(batch);
  hipLaunchKernelGGL(rank1_colsum_kernel<T>, dim3(static_cast<unsigned>(ceil_div(a.cols, kColTile)), nb),
                     dim3(kColTile * kColRows), 0, st, a);
  int rc = check_launch("rank1_apply column sums");
  if (rc) return rc;
  // Four waves per row from 256 columns on (four columns per lane with one),
  // as long as the rows alone don't fill the device many times over.
  if (a.cols >= 256 && a.rows <= 65536)
    hipLaunchKernelGGL((rank1_row_kernel<T, 4>), dim3(static_cast<unsigned>(a.rows), nb), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((rank1_row_kernel<T, 1>), dim3(static_cast<unsigned>(ceil_div(a.rows, 4)), nb), dim3(256), 0,
                       st, a);
  return check_launch("rank1_apply rows");
}

// ---------------------------------------------------- inverse sqrt ---
template <typename T>
__device__ __forceinline__ T rsqrt_t(T v);
template <>
__device__ __forceinline__ float rsqrt_t<float>(float v) { return rsqrtf(v); }
template <>
__device__ __forceinline__ double rsqrt_t<double>(double v) { return 1.0 / sqrt(v); }

template <typename T>
constexpr T tiny_t() { return sizeof(T) == 4 ? static_cast<T>(FLT_MIN) : static_cast<T>(DBL_MIN); }

// One block of 1024 threads per vector.  Means and sum z^2 in FP64,
// rounded to T where the reference holds them in T.
template <typename T>
__global__ void __launch_bounds__(1024) inverse_sqrt_kernel(int kind, const T *second, const T *mean, int64_t n,
                                                             T *inv, T *z, T *kappa) {
  __shared__ double scratch[16];
  double s = 0.0;
  for (int64_t c = threadIdx.x; c < n; c += blockDim.x) s += static_cast<double>(second[c]);
  const T m = static_cast<T>(block_sum(s, scratch) / static_cast<double>(n));
  if (kind == 0) {
    const T floor = m * static_cast<T>(1e-6);
    const T den = m > tiny_t<T>() ? m : tiny_t<T>();
    for (int64_t c = threadIdx.x; c < n; c += blockDim.x) {
      const T v = second[c] > floor ? second[c] : floor;
      const T r = v / den;
      inv[c] = rsqrt_t<T>(r > static_cast<T>(1e-6) ? r : static_cast<T>(1e-6));
    }
    return;
  }
  const T q = m > tiny_t<T>() ? m : tiny_t<T>();
  const T sq = sqrt(q);
  double zpart = 0.0;
  for (int64_t c = threadIdx.x; c < n; c += blockDim.x) {
    const T mc = mean[c];
    T var = second[c] - mc * mc;
    var = var > static_cast<T>(0) ? var : static_cast<T>(0);
    const T r = var / q;
    const T iv = rsqrt_t<T>(r > static_cast<T>(1e-6) ? r : static_cast<T>(1e-6));
    const T zc = iv * (mc / sq);
    inv[c] = iv;
    z[c] = zc;
    zpart += static_cast<double>(zc) * static_cast<double>(zc);
  }
  const T zz = static_cast<T>(block_sum(zpart, scratch));
  if (threadIdx.x == 0) {
    const T rho = sqrt(static_cast<T>(1) + zz);
    kappa[0] = static_cast<T>(-1) / (rho * (rho + static_cast<T>(1)));
  }
}

// ------------------------------------------------------------- graft ---
// out = x * sqrt(rows) / max(||x||_F, FLT_MIN) (zero stays zero).
// Pass 1: per-block partial sums of squares; pass 2: scale.
__global__ void __launch_bounds__(256) graft_partial_kernel(const float *x, int64_t n, double *parts) {
  __shared__ double scratch[16];
  double s = 0.0;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < n; e += static_cast<int64_t>(gridDim.x) * 256) {
    const double v = x[e];
    s += v * v;
  }
  s = block_sum(s, scratch);
  if (threadIdx.x == 0) parts[blockIdx.x] = s;
}

__global__ void __launch_bounds__(256) graft_scale_kernel(const float *x, float *out, int64_t n, const double *parts,
                                                          int nparts, float sqrt_rows) {
  __shared__ double bcast;
  if (threadIdx.x < 64) {
    double s = 0.0;
    for (int k = threadIdx.x; k < nparts; k += 64) s += parts[k];
    s = wave_sum(s);
    if (threadIdx.x == 0) bcast = s;
  }
  __syncthreads();
  const double n2 = bcast;
  const float scale = n2 > 0.0 ? sqrt_rows / fmaxf(static_cast<float>(sqrt(n2)), FLT_MIN) : 0.f;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < n; e += static_cast<int64_t>(gridDim.x) * 256)
    out[e] = x[e] * scale;
}

}  // namespace smx

using namespace smx;

extern "C" int smx_inverse_sqrt(int kind, int dtype, const void *second, const void *mean, int64_t n, void *inv,
                                void *z, void *kappa, void *stream) {
  SMX_REQUIRE(kind == 0 || kind == 1, SMX_EINVAL, "inverse_sqrt: kind must be 0 (diagonal) or 1 (rank-one)");
  SMX_REQUIRE(dtype == SMX_F32 || dtype == SMX_F64, SMX_EDTYPE, "inverse_sqrt: dtype must be f32 or f64");
  SMX_REQUIRE(n >= 1, SMX_ESHAPE, "inverse_sqrt: n must be >= 1");
  SMX_REQUIRE(second && inv, SMX_EINVAL, "inverse_sqrt: null pointer");
  SMX_REQUIRE(kind == 0 || (mean && z && kappa), SMX_EINVAL, "inverse_sqrt: rank-one needs mean, z and kappa");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == SMX_F32)
    hipLaunchKernelGGL(inverse_sqrt_kernel<float>, dim3(1), dim3(1024), 0, st, kind,
                       static_cast<const float *>(second), static_cast<const float *>(mean), n,
                       static_cast<float *>(inv), static_cast<float *>(z), static_cast<float *>(kappa));
  else
    hipLaunchKernelGGL(inverse_sqrt_kernel<double>, dim3(1), dim3(1024), 0, st, kind,
                       static_cast<const double *>(second), static_cast<const double *>(mean), n,
                       static_cast<double *>(inv), static_cast<double *>(z), static_cast<double *>(kappa));
  return check_launch("inverse_sqrt");
}

extern "C" int smx_rank1_apply_shared(int dtype, const void *x, void *out, int64_t batch, int64_t rows, int64_t cols,
                                      const void *li, const void *lz, const void *lc, const void *ri, const void *rz,
                                      const void *rc, int shared, int order, double *work, void *stream) {
  SMX_REQUIRE(shared >= 0 && shared <= 3, SMX_EINVAL, "rank1_apply: shared must be in [0, 3]");
  const int64_t lb = shared & 1 ? 0 : 1, rb = shared & 2 ? 0 : 1;
  SMX_REQUIRE(dtype == SMX_F32 || dtype == SMX_F64, SMX_EDTYPE, "rank1_apply: dtype must be f32 or f64");
  SMX_REQUIRE(x && out && li && lz && lc && ri && rz && rc && work, SMX_EINVAL, "rank1_apply: null pointer");
  SMX_REQUIRE(order == 0 || order == 1, SMX_EINVAL, "rank1_apply: order must be 0 (whiten) or 1 (mapback)");
  SMX_REQUIRE(batch >= 0 && rows >= 1 && cols >= 1 && batch <= 65535, SMX_ESHAPE, "rank1_apply: bad shape");
  SMX_REQUIRE(ceil_div(rows * cols, 256) <= 0x7fffffff, SMX_ESHAPE, "rank1_apply: matrix too large");
  SMX_REQUIRE(out != x, SMX_EINVAL, "rank1_apply: out must not alias x");
  if (batch == 0) return SMX_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  double *t = work;
  if (dtype == SMX_F32) {
    Rank1Args<float> a{static_cast<const float *>(x), static_cast<float *>(out), rows, cols,
                       static_cast<const float *>(li), static_cast<const float *>(lz), static_cast<const float *>(lc),
                       static_cast<const float *>(ri), static_cast<const float *>(rz), static_cast<const float *>(rc),
                       t, order, lb, rb};
    return launch_rank1(a, batch, st);
  }
  Rank1Args<double> a{static_cast<const double *>(x), static_cast<double *>(out), rows, cols,
                      static_cast<const double *>(li), static_cast<const double *>(lz),
                      static_cast<const double *>(lc), static_cast<const double *>(ri),
                      static_cast<const double *>(rz), static_cast<const double *>(rc), t, order, lb, rb};
  return launch_rank1(a, batch, st);
}

extern "C" int smx_rank1_apply(int dtype, const void *x, void *out, int64_t batch, int64_t rows, int64_t cols,
                               const void *li, const void *lz, const void *lc, const void *ri, const void *rz,
                               const void *rc, int order, double *work, void *stream) {
  return smx_rank1_apply_shared(dtype, x, out, batch, rows, cols, li, lz, lc, ri, rz, rc, 0, order, work, stream);
}

extern "C" int smx_graft(const float *x, float *out, int64_t n, int64_t output_rows, double *work, int32_t work_len,
                         void *stream) {
  SMX_REQUIRE(x && out && work, SMX_EINVAL, "graft: null pointer");
  SMX_REQUIRE(n >= 0 && output_rows >= 0 && work_len >= 1, SMX_ESHAPE, "graft: bad size");
  if (n == 0) return SMX_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nb = static_cast<int>(std::min<int64_t>(work_len, std::min<int64_t>(1024, ceil_div(n, 256))));
  hipLaunchKernelGGL(graft_partial_kernel, dim3(nb), dim3(256), 0, st, x, n, work);
  int rc = check_launch("graft partial");
  if (rc) return rc;
  hipLaunchKernelGGL(graft_scale_kernel, dim3(nb), dim3(256), 0, st, x, out, n, work, nb,
                     static_cast<float>(std::sqrt(static_cast<double>(output_rows))));
  return check_launch("graft scale");
}
