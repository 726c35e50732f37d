// Stand-alone S8 polar map on a strided batch (the module-level _s8_fp32
// helper of sandmuon/optimizer.py:69-93): load -> five stages -> store.
#include "s8.h"

#include <algorithm>
#include <memory>
#include <vector>

namespace smx {

struct S8IoArgs {
  S8Class k;
  const float *x;
  float *out;
  int64_t rows, cols;          // input (= output) shape per matrix
  int64_t sb, sr, sc;          // element strides: batch, row, col
  int32_t planes;              // iterate stored as BF16 planes (comp mode)
};

// Load: 64x64 tiles of the padded parameter layout (input layout) into the
// oriented iterate x0 (a tiled operand), directly or transposed through LDS
// for transposed parameters, with the input's sum of squares from the same
// read: a block takes tiles blockIdx.x, blockIdx.x + gridDim.x, ... of one
// matrix and leaves one FP64 partial.  Bound by HBM (8 bytes per padded
// element): a block per tile keeps every CU reading, where the sum of
// squares as a pass of one block per matrix was the longest launch of the
// call (nine 3072 x 768 matrices: 3722 us for that pass and 38 for the
// tiles, 44 for this kernel).  VEC: 16-byte loads (unit column stride,
// rows on 16-byte boundaries).  grid = (blocks, batch), block 256.
template <bool VEC>
__global__ void __launch_bounds__(256) s8_load_kernel(S8IoArgs a) {
  __shared__ float tile[64][65];
  __shared__ double scratch[16];
  const S8Mat M{a.k, static_cast<int32_t>(blockIdx.y)};
  const float *x = a.x + static_cast<int64_t>(blockIdx.y) * a.sb;
  float *pl = M.flip() ? nullptr : M.x0();
  float *tl = M.flip() ? M.x0() : nullptr;
  const int64_t ppad = M.pcol_pad(), rpad = M.prow_pad();
  const int64_t tiles_c = ppad / 64, tiles = tiles_c * (rpad / 64);
  const int t = threadIdx.x, lc = (t & 15) * 4;
  double s = 0.0;
  for (int64_t tix = blockIdx.x; tix < tiles; tix += gridDim.x) {
    const int64_t i0 = (tix / tiles_c) * 64, j0 = (tix % tiles_c) * 64;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int lr = (t >> 4) + 16 * q;
      const int64_t i = i0 + lr, j = j0 + lc;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      if (VEC) {
        if (i < a.rows && j < a.cols) {  // cols is a multiple of 4
          const float4 w = *reinterpret_cast<const float4 *>(x + i * a.sr + j);
          v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i < a.rows && j + e < a.cols) v[e] = x[i * a.sr + (j + e) * a.sc];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = fma(static_cast<double>(v[e]), static_cast<double>(v[e]), s);
        if (tl) tile[lr][lc + e] = v[e];
      }
      if (pl) put_operand4(pl, tiled_index(i, j, ppad), v, a.planes != 0);
    }
    if (!tl) continue;  // uniform per block
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int lr = (t >> 4) + 16 * q;
      const float v[4] = {tile[lc][lr], tile[lc + 1][lr], tile[lc + 2][lr], tile[lc + 3][lr]};
      put_operand4(tl, tiled_index(j0 + lr, i0 + lc, rpad), v, a.planes != 0);
    }
    __syncthreads();
  }
  s = block_sum(s, scratch);
  if (t == 0) M.fro()[blockIdx.x] = s;
}

// The input's sum of squares: the load's `n` partials in a fixed order ->
// the matrix's kCstFro.  grid = batch, block 256.
__global__ void __launch_bounds__(256) s8_load_total_kernel(S8IoArgs a, int32_t n) {
  __shared__ double scratch[16];
  const S8Mat M{a.k, static_cast<int32_t>(blockIdx.x)};
  double s = 0.0;
  for (int32_t i = threadIdx.x; i < n; i += 256) s += M.fro()[i];
  s = block_sum(s, scratch);
  if (threadIdx.x == 0) {
    M.cst()[kCstFro] = s;
    M.cst()[kCstWide] = 0.0;
  }
}

// Store: final iterate (parameter layout) -> out (strided), four columns
// per thread; VEC: 16-byte stores.  (A result whose padded shape is `out`'s
// own is written there by the last stage: `direct` of smx_s8.)
// grid = (ceil(rows * ceil(cols / 4) / 256), batch).
template <bool VEC>
__global__ void __launch_bounds__(256) s8_store_kernel(S8IoArgs a) {
  const S8Mat M{a.k, static_cast<int32_t>(blockIdx.y)};
  const float *q = M.result();
  const int64_t c4 = ceil_div(a.cols, 4);
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= a.rows * c4) return;
  const int64_t i = e / c4, j = (e % c4) * 4;
  const float4 w = *reinterpret_cast<const float4 *>(q + i * M.pcol_pad() + j);
  float *o = a.out + static_cast<int64_t>(blockIdx.y) * a.sb + i * a.sr;
  if (VEC) {
    *reinterpret_cast<float4 *>(o + j) = w;
    return;
  }
  const float v[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (j + k < a.cols) o[(j + k) * a.sc] = v[k];
}

}  // namespace smx

using namespace smx;

static bool plan_single(int64_t batch, int64_t rows, int64_t cols, int mode, char *base, S8Plan &plan) {
  const bool flip = rows > cols;
  std::vector<int64_t> r(batch, flip ? cols : rows), c(batch, flip ? rows : cols);
  std::unique_ptr<bool[]> f(new bool[batch]);
  for (int64_t i = 0; i < batch; ++i) f[i] = flip;
  std::vector<int32_t> cls(batch), slot(batch);
  return plan_s8(r.data(), c.data(), f.get(), nullptr, static_cast<int32_t>(batch), mode, base, plan, cls.data(),
                 slot.data());
}

extern "C" size_t smx_s8_workspace_bytes(int64_t batch, int64_t rows, int64_t cols, int mode) {
  if (batch < 1 || rows < 1 || cols < 1) return 0;
  S8Plan plan;
  plan_single(batch, rows, cols, mode, nullptr, plan);
  return plan.bytes;
}

extern "C" int smx_s8(const float *x, float *out, int64_t batch, int64_t rows, int64_t cols, int64_t batch_stride,
                      int64_t row_stride, int64_t col_stride, int mode, void *workspace, size_t workspace_bytes,
                      void *stream) {
  SMX_REQUIRE(x && out, SMX_EINVAL, "s8: null pointer");
  SMX_REQUIRE(mode == SMX_S8_FP32 || mode == SMX_S8_COMP_BF16 || mode == SMX_S8_MIXED, SMX_EINVAL,
              "s8: unknown mode");
  SMX_REQUIRE(batch >= 0 && rows >= 0 && cols >= 0, SMX_ESHAPE, "s8: negative shape");
  SMX_REQUIRE(batch <= 65535, SMX_ESHAPE, "s8: batch must be <= 65535");
  if (batch == 0 || rows == 0 || cols == 0) return SMX_OK;
  SMX_REQUIRE(workspace, SMX_EINVAL, "s8: null workspace");
  SMX_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 256 == 0, SMX_EALIGN, "s8: workspace must be 256-byte aligned");
  S8Plan plan;
  plan_single(batch, rows, cols, mode, static_cast<char *>(workspace), plan);
  SMX_REQUIRE(workspace_bytes >= plan.bytes, SMX_EWORKSPACE, "s8: workspace too small");
  hipStream_t st = static_cast<hipStream_t>(stream);
  S8IoArgs a{};
  a.k = plan.layout.cls[0];
  a.x = x;
  a.out = out;
  a.rows = rows;
  a.cols = cols;
  a.sb = batch_stride;
  a.sr = row_stride;
  a.sc = col_stride;
  a.planes = mode != SMX_S8_FP32;  // stage 1 reads X0 compensated in both BF16 modes
  // Four columns at a time where every row starts on a 16-byte boundary.
  const bool vec_rows = a.sc == 1 && cols % 4 == 0 && a.sr % 4 == 0 && a.sb % 4 == 0;
  const bool vec_in = vec_rows && reinterpret_cast<uintptr_t>(x) % 16 == 0;
  const bool vec_out = vec_rows && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  // A result of unpadded shape goes straight to `out`, which takes the
  // place of the buffer that the last stage writes (S8Mat::result).  That
  // buffer also holds an iterate while x is still read, so `out` must not
  // overlap x.
  S8Class &K = plan.layout.cls[0];
  const size_t bytes = static_cast<size_t>(batch) * rows * cols * sizeof(float);
  const uintptr_t xa = reinterpret_cast<uintptr_t>(x), oa = reinterpret_cast<uintptr_t>(out);
  const bool direct = K.r == K.rp && K.c == K.cp && a.sc == 1 && a.sr == cols && (batch == 1 || a.sb == rows * cols) &&
                      oa % 256 == 0 && (oa + bytes <= xa || xa + bytes <= oa);
  if (direct) (K.n_flip ? K.xf : K.gs ? K.x0 : K.x1) = out;
  a.k = K;
  const S8Mat M0{a.k, 0};
  const int64_t tiles = (M0.prow_pad() / 64) * (M0.pcol_pad() / 64);
  const int32_t blocks = static_cast<int32_t>(std::min<int64_t>(tiles, K.parts));
  const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(batch));
  if (vec_in) hipLaunchKernelGGL(s8_load_kernel<true>, grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL(s8_load_kernel<false>, grid, dim3(256), 0, st, a);
  int rc = check_launch("s8 load");
  if (rc) return rc;
  hipLaunchKernelGGL(s8_load_total_kernel, dim3(static_cast<unsigned>(batch)), dim3(256), 0, st, a, blocks);
  rc = check_launch("s8 load total");
  if (rc) return rc;
  rc = run_s8_stages(plan.layout, st);
  if (rc || direct) return rc;
  const dim3 sgrid(static_cast<unsigned>(ceil_div(rows * ceil_div(cols, 4), 256)), static_cast<unsigned>(batch));
  if (vec_out) hipLaunchKernelGGL(s8_store_kernel<true>, sgrid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL(s8_store_kernel<false>, sgrid, dim3(256), 0, st, a);
  return check_launch("s8 store");
}
