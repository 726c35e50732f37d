// The S8 map of small matrices: one block runs all five stages of one
// matrix in LDS (sandmuon/optimizer.py:69-93), in place of the 15-23
// launches of s8.hip on operands padded to 256.
//
// A class is small when its iterate and Gram, padded to 16, fit one block's
// LDS in FP32 (small_bytes) with at most kSmallTiles row tiles.  Every
// product runs on FP32 MFMAs (v_mfma_f32_16x16x4_f32) whatever the mode: no
// operand is rounded below FP32 but the input, which the other modes hand over
// as BF16 hi + lo (16-17 bits).  From stage 2 on the Gram is held as H = G
// - I and P formed from it (as kS8Pair does in s8.hip).  Bound by latency
// (chains of dependent MFMAs and LDS reads between barriers), not by the
// matrix cores' rate, up to about 64 rows.  The S8 of the 12 matrices of a
// toy GPT (32 x 32 to 128 x 32) takes 31 us in place of 220 us in launches of
// 64 x 64 and 128 x 128 tiles; 24 matrices of 72 x 200 85 us a call in place
// of 220.
//
// Stage k on X (r x c, r <= c, rows in LDS at a pitch of 4 words more than a
// multiple of 16, so that 16 lanes reading 16 bytes of 16 rows hit distinct
// banks):
//   Gram    G = X X^T: upper-triangle 16 x 16 tiles over the block's waves;
//           where there are fewer tiles than waves, K is split too and the
//           partial tiles are added in order through LDS
//   square  a wave per 16 columns: P = c G G + b G + a I in registers, then,
//           after a barrier, over G (stage 1: G G, its Frobenius norm over
//           the block, then P1)
//   apply   a wave per 16 columns of X: X' = P X over those columns in place
//           (they depend on no other columns)
#include "s8.h"

#include <algorithm>
#include <cmath>

namespace smx {

constexpr int kSmallThreads = 1024, kSmallWaves = kSmallThreads / 64;
constexpr int kSmallTiles = 8;  // row tiles of 16: the accumulators a wave holds per column tile
constexpr int kSmallPartBytes = kSmallWaves * 256 * 4;  // a partial Gram tile per wave
constexpr int kSmallLds = 64 << 10, kSmallLdsBig = 158 << 10;  // two blocks per CU, or one

struct SmallArgs {
  S8Layout L;
  int32_t start[kMaxClasses + 1];  // first block of each class (no blocks: not small)
};

__host__ __device__ inline int small_pitch(int64_t n) { return static_cast<int>(round_up(n, 16)) + 4; }
// X, G and the partial tiles.
__host__ __device__ inline int64_t small_bytes(const S8Class &k) {
  const int64_t r16 = round_up(k.r, 16);
  return 4 * r16 * (small_pitch(k.c) + small_pitch(k.r)) + kSmallPartBytes;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// acc += A B over K = 16: lane l holds A[l & 15][4 (l >> 4) + q] and
// B[4 (l >> 4) + q][l & 15] for q = 0..3 (the same permutation of K for
// both).  acc[e] is element [4 (l >> 4) + e][l & 15].
__device__ __forceinline__ void mma16(const f32x4 &a, const f32x4 &b, f32x4 &acc) {
#pragma unroll
  for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[q], acc, 0, 0, 0);
}

// The block's class and slot.
__device__ __forceinline__ S8Mat small_find(const SmallArgs &args, int blk) {
  int ci = 0;
  while (ci + 1 < args.L.n_classes && blk >= args.start[ci + 1]) ++ci;
  return S8Mat{args.L.cls[ci], blk - args.start[ci]};
}

// The result X (pitch px) in parameter layout, and for the matrix step each
// row's sums of Q z, (a Q)^2 and (a Q)(a z) as its first strip (zeros in the
// others).
__device__ __forceinline__ void small_store(const SmallArgs &args, const float *X, int px) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int blk = blockIdx.x;
  asm volatile("" : "+s"(blk));  // found again here: the class's fields are not held over the stages
  const S8Mat M = small_find(args, blk);
  const bool flip = M.flip(), rsum = args.L.rowsums != 0;
  const int prow = static_cast<int>(M.prow()), pcol = static_cast<int>(M.pcol());
  const int sr = flip ? 1 : px, sc = flip ? px : 1;
  const int ld = static_cast<int>(M.pcol_pad()), ppad = static_cast<int>(M.prow_pad());
  SMX_GLOBAL float *out = (SMX_GLOBAL float *)M.result();
  const SMX_GLOBAL float *acol = rsum ? (const SMX_GLOBAL float *)M.acol() : nullptr;
  const SMX_GLOBAL float *zcol = rsum ? (const SMX_GLOBAL float *)M.zcol() : nullptr;
  SMX_GLOBAL float *mr = (SMX_GLOBAL float *)M.mrp(0);
  const int64_t msz = M.mrp_size();
  const int strips = static_cast<int>(M.strips());
  for (int p = wave; p < prow; p += kSmallWaves) {
    float s[3] = {0.f, 0.f, 0.f};
    for (int j = lane; j < pcol; j += 64) {
      const float q = X[p * sr + j * sc];
      out[static_cast<int64_t>(p) * ld + j] = q;
      if (rsum) {
        const float a = acol[j], z = zcol ? zcol[j] : 0.f, aq = a * q;
        s[0] = fmaf(q, z, s[0]);
        s[1] = fmaf(aq, aq, s[1]);
        s[2] = fmaf(aq, a * z, s[2]);
      }
    }
    if (rsum) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float v = wave_sum(s[k]);
        for (int t = lane; t < strips; t += 64) mr[k * msz + static_cast<int64_t>(t) * ppad + p] = t == 0 ? v : 0.f;
      }
    }
  }
}

// One matrix of R row tiles.
template <int R>
__device__ __forceinline__ void small_body(const SmallArgs &args, float *lds, double *scratch) {
  const S8Mat M = small_find(args, blockIdx.x);
  const S8Class &K = *M.kp();
  const int r = static_cast<int>(K.r), c = static_cast<int>(K.c);
  const int C = (c + 15) / 16;  // column tiles
  const int px = small_pitch(c);
  constexpr int pg = 16 * R + 4;
  float *const X = lds, *const G = X + 16 * R * px, *const part = G + 16 * R * pg;
  const int lane = threadIdx.x & 63, wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;  // the lane's row or column of a tile, its quarter of K

  // X = V / ||V||, from the tiled operand form (its padding holds zeros).
  double fro2 = M.cst()[kCstFro];
  asm volatile("" : "+v"(fro2));  // held over the Gram in vector registers: the scalar ones are all taken
  const float inv_fro = fro2 > 0.0 ? static_cast<float>(1.0 / sqrt(fro2)) : 0.f;
  const bool planes = args.L.mode != SMX_S8_FP32;
  {
    const SMX_GLOBAL char *x0 = (const SMX_GLOBAL char *)M.x0();
    const int quads = 16 * R * C * 4;  // quarters of the rows' K groups
    for (int i = threadIdx.x; i < quads; i += kSmallThreads) {
      const int qt = i & 3, row = (i >> 2) % (16 * R), grp = (i >> 2) / (16 * R);
      const SMX_GLOBAL char *p = x0 + 4 * tiled_index(row, 16 * grp, K.cp);
      f32x4 v;
      if (planes) {
        const u32x2v h = *reinterpret_cast<const SMX_GLOBAL u32x2v *>(p + 8 * qt);
        const u32x2v l = *reinterpret_cast<const SMX_GLOBAL u32x2v *>(p + 32 + 8 * qt);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          v[2 * e] = __uint_as_float(h[e] << 16) + __uint_as_float(l[e] << 16);
          v[2 * e + 1] = __uint_as_float(h[e] & 0xffff0000u) + __uint_as_float(l[e] & 0xffff0000u);
        }
      } else {
        v = *reinterpret_cast<const SMX_GLOBAL f32x4 *>(p + 16 * qt);
      }
      *reinterpret_cast<f32x4 *>(X + row * px + 16 * grp + 4 * qt) = v * inv_fro;
    }
  }
  __syncthreads();

  constexpr int tiles = R * (R + 1) / 2;
  constexpr int split = kSmallWaves / tiles > 1 ? kSmallWaves / tiles : 1;  // waves per Gram tile
  for (int stage = 1; stage <= 5; ++stage) {
    int wave = wave_id;
    asm volatile("" : "+s"(wave));  // what derives from it is not kept over the stages (scalar registers)
    // subtracts I from the lane's elements of a diagonal tile of the Gram
    auto shift = [&](f32x4 &acc, int ti, int tj) {
      if (stage == 1 || ti != tj || 16 * ti + n >= r) return;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * g + e == n) acc[e] -= 1.f;
    };
    // ---- Gram
    for (int w = wave; w < tiles * split; w += kSmallWaves) {
      const int t = w / split, s = w % split;
      int ti = 0, rem = t;
      while (rem >= R - ti) { rem -= R - ti; ++ti; }
      const int tj = ti + rem;
      const float *a = X + (16 * ti + n) * px + 4 * g, *b = X + (16 * tj + n) * px + 4 * g;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      const int k1 = C * (s + 1) / split;
      for (int k = C * s / split; k < k1; ++k)
        mma16(*reinterpret_cast<const f32x4 *>(a + 16 * k), *reinterpret_cast<const f32x4 *>(b + 16 * k), acc);
      if (split > 1) {
        *reinterpret_cast<f32x4 *>(part + 256 * w + 4 * lane) = acc;
      } else {
        shift(acc, ti, tj);
        *reinterpret_cast<f32x4 *>(G + (16 * tj + n) * pg + 16 * ti + 4 * g) = acc;
        if (ti != tj)
#pragma unroll
          for (int e = 0; e < 4; ++e) G[(16 * ti + 4 * g + e) * pg + 16 * tj + n] = acc[e];
      }
    }
    __syncthreads();
    if (split > 1) {
      for (int t = wave; t < tiles; t += kSmallWaves) {
        int ti = 0, rem = t;
        while (rem >= R - ti) { rem -= R - ti; ++ti; }
        const int tj = ti + rem;
        f32x4 acc = *reinterpret_cast<const f32x4 *>(part + 256 * t * split + 4 * lane);
        for (int s = 1; s < split; ++s) acc += *reinterpret_cast<const f32x4 *>(part + 256 * (t * split + s) + 4 * lane);
        shift(acc, ti, tj);
        *reinterpret_cast<f32x4 *>(G + (16 * tj + n) * pg + 16 * ti + 4 * g) = acc;
        if (ti != tj)
#pragma unroll
          for (int e = 0; e < 4; ++e) G[(16 * ti + 4 * g + e) * pg + 16 * tj + n] = acc[e];
      }
      __syncthreads();
    }
    // ---- square: the wave's 16 columns of G G, and of P
    f32x4 sq[R];
#pragma unroll
    for (int i = 0; i < R; ++i) sq[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (wave < R) {
#pragma unroll 2
      for (int k = 0; k < R; ++k) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(G + (16 * wave + n) * pg + 16 * k + 4 * g);
#pragma unroll
        for (int i = 0; i < R; ++i)
          if (i < R) mma16(*reinterpret_cast<const f32x4 *>(G + (16 * i + n) * pg + 16 * k + 4 * g), b, sq[i]);
      }
    }
    float s2 = 1.f, xscale = 1.f;  // stage 1: the Schatten scale squared, and 1/s of the apply
    if (stage == 1) {
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum = fma(static_cast<double>(sq[i][e]), static_cast<double>(sq[i][e]), sum);
      sum = block_sum(sum, scratch);
      const bool ok = fro2 > 0.0 && sum > 0.0;
      const float s = ok ? fmaxf(static_cast<float>(kS8Margin * pow(sum, 0.125)), 1e-30f) : 1.f;
      s2 = s * s;
      xscale = ok ? 1.0f / s : 0.f;
    }
    const double *co = kS8Coefficients[stage - 1];
    const float cc = static_cast<float>(co[2]);
    const float cb = static_cast<float>(stage == 1 ? co[1] : co[1] + 2 * co[2]);
    const float ca = static_cast<float>(stage == 1 ? co[0] : co[0] + co[1] + co[2]);
    const float is2 = 1.0f / s2, is4 = 1.0f / (s2 * s2);
    if (wave < R) {
      // element e of tile i is on the diagonal of P where i = wave, e = de;
      // kept opaque, or the masks of every stage are hoisted and spill
      int de = 16 * wave + n < r ? n - 4 * g : -1;
      asm volatile("" : "+v"(de));
#pragma unroll
      for (int i = 0; i < R; ++i) {
        // (G and G G are symmetric: the tile's transpose is read and written)
        const f32x4 gv = *reinterpret_cast<const f32x4 *>(G + (16 * wave + n) * pg + 16 * i + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float eye = i == wave && de == e ? ca : 0.f;
          sq[i][e] = (eye + (cb * gv[e]) * is2) + (cc * sq[i][e]) * is4;
        }
      }
    }
    __syncthreads();
    if (wave < R) {
#pragma unroll
      for (int i = 0; i < R; ++i)
        *reinterpret_cast<f32x4 *>(G + (16 * wave + n) * pg + 16 * i + 4 * g) = sq[i];
    }
    __syncthreads();
    // ---- apply: columns 16 t .. 16 t + 15 of X, in place
    for (int t = wave; t < C; t += kSmallWaves) {
      f32x4 acc[R];
#pragma unroll
      for (int i = 0; i < R; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      float *x = X + 16 * t + n;
#pragma unroll 2
      for (int k = 0; k < R; ++k) {
        f32x4 b;
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = x[(16 * k + 4 * g + q) * px];
#pragma unroll
        for (int i = 0; i < R; ++i)
          if (i < R) mma16(*reinterpret_cast<const f32x4 *>(G + (16 * i + n) * pg + 16 * k + 4 * g), b, acc[i]);
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[(16 * i + 4 * g + e) * px] = acc[i][e] * xscale;
      }
    }
    __syncthreads();
  }

  // The result in parameter layout, and for the matrix step each row's sums
  // of Q z, (a Q)^2 and (a Q)(a z) as its first strip (zeros in the others).
  small_store(args, X, px);
}

template <int R, int BYTES>
__global__ void __launch_bounds__(kSmallThreads) s8_small_kernel(SmallArgs args) {
  __shared__ __attribute__((aligned(16))) float lds[BYTES / 4];
  __shared__ double scratch[16];
  small_body<R>(args, lds, scratch);
}

template <int R>
static void launch_small(int64_t bytes, int32_t blocks, const SmallArgs &a, hipStream_t st) {
  if (bytes <= kSmallLds)
    hipLaunchKernelGGL((s8_small_kernel<R, kSmallLds>), dim3(blocks), dim3(kSmallThreads), 0, st, a);
  else
    hipLaunchKernelGGL((s8_small_kernel<R, kSmallLdsBig>), dim3(blocks), dim3(kSmallThreads), 0, st, a);
}

bool s8_small(const S8Class &k) {
  return !k.low && k.r <= 16 * kSmallTiles && small_bytes(k) <= kSmallLdsBig;
}

int run_s8_small(const S8Layout &Lay, hipStream_t st, double &flops) {
  for (int R = 1; R <= kSmallTiles; ++R) {  // one launch for the classes of R row tiles
    SmallArgs a{};
    a.L = Lay;
    int32_t blocks = 0;
    int64_t bytes = 0;
    for (int i = 0; i < Lay.n_classes; ++i) {
      const S8Class &k = Lay.cls[i];
      a.start[i] = blocks;
      if (!k.count || !s8_small(k) || ceil_div(k.r, 16) != R) continue;
      blocks += k.count;
      bytes = std::max(bytes, small_bytes(k));
      const double r = 16.0 * R, c = static_cast<double>(round_up(k.c, 16));
      flops += 5.0 * k.count * (r * (r + 16) * c + 2 * r * r * r + 2 * r * r * c);
    }
    for (int i = Lay.n_classes; i <= kMaxClasses; ++i) a.start[i] = blocks;
    if (!blocks) continue;
    switch (R) {
      case 1: launch_small<1>(bytes, blocks, a, st); break;
      case 2: launch_small<2>(bytes, blocks, a, st); break;
      case 3: launch_small<3>(bytes, blocks, a, st); break;
      case 4: launch_small<4>(bytes, blocks, a, st); break;
      case 5: launch_small<5>(bytes, blocks, a, st); break;
      case 6: launch_small<6>(bytes, blocks, a, st); break;
      case 7: launch_small<7>(bytes, blocks, a, st); break;
      default: launch_small<kSmallTiles>(bytes, blocks, a, st); break;
    }
    const int rc = check_launch("s8 small");
    if (rc) return rc;
  }
  return SMX_OK;
}

}  // namespace smx
