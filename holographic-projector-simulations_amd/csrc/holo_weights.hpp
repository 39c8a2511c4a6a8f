// The weights of the 16-row lattice kernels as MFMA operands: device code shared
// by k_grid16_weights (holo_grid.hip) and k_pair_prep (holo_pairs.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "holo_device.hpp"
#include "holo_internal.hpp"

namespace holo {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));

constexpr int kGridWaves = kBlock / 64;
// f16 scales of the correction operands: the weight side carries k_a kCrossW W
// (and k_a^2 kCross2W W), the column side the inverse, so that both sides stay
// in f16's normal range from a few cm to about a metre.
constexpr float kCrossW = 0x1p-4f;
constexpr float kCross2W = 0x1p-8f;

// x = hi + lo in f16: hi is x rounded to 11 significant bits (ties away from
// zero) by integer arithmetic, so hi is exact in f16 for |x| >= 2^-14 and
// every conversion instruction yields the same hi; lo = x - hi is exact in
// FP32 and |lo| <= 2^-11 |x|.  (Splitting as lo = x - (float)(half)x is not
// safe: the compiler may fold the product that made x into the f16
// conversion -- one rounding instead of two -- for one use of hi and not for
// another, and at exact ties hi + lo is then off by one f16 ulp.)
__device__ __forceinline__ void split_f16(float x, _Float16& hi, _Float16& lo) {
  const float h =
      __builtin_bit_cast(float, (__builtin_bit_cast(uint32_t, x) + 0x1000u) & 0xffffe000u);
  hi = (_Float16)h;
  lo = (_Float16)(x - h);
}

// MFMA operands of the 16 x 16 tiles' weights, one wave per tile: for row
// block rb, wq[(6t + 3rb + q) * 64 + lane] holds, for lane l = 16 g + i,
// row i = 2a' + c (a = 8 rb + a') and columns 4g .. 4g + 3 (re, im) of the real
// form of W / tscale split into f16 hi (q = 0) and lo (q = 1), and of
// i k_a kCrossW W / tscale (q = 2, its f16 hi part).  wqn (nullable), the
// near-field GEMM's extra operands: wqn[(4t + 2rb + q) * 64 + lane] holds the
// lo part of i k_a kCrossW W / tscale (q = 0) and k_a^2 kCross2W W / tscale in
// the real form of W (q = 1).  The weights come from the caller's (w0, w1, wf: as
// launch_tile_weights) through perm, 256 slots per tile, slot 16 a + b, and go to
// wc as well, with those of the n_tail slots after the tiles (the workgroups
// beyond the tiles').
// group (1, 2 or 4): tiles group T .. group T + group - 1 (the halves of a
// 16 x 32 tile, the quarters of a 16 x 64 one) share one tscale, the power of
// two above the largest of their largest components.
// block: the workgroup's index among the grid16_weight_blocks of the launch.
__device__ __forceinline__ void grid16_weights(const Grid16Prep& a, uint32_t block) {
  const uint32_t tile_blocks = (a.n_tiles + kGridWaves - 1) / kGridWaves;
  if (block >= tile_blocks) {  // the whole workgroup
    const uint32_t k = (block - tile_blocks) * kBlock + threadIdx.x;
    if (k < a.n_tail) {
      const size_t at = (size_t)a.n_tiles * 256 + k;
      a.wc[at] = slot_weight(a.wf, a.w0, a.w1, a.perm[at]);
    }
    return;
  }
  __shared__ float s_max[kGridWaves];
  __shared__ float2 s_w[kGridWaves][256];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t t = block * kGridWaves + wv;
  const uint32_t i = lane & 15, g = lane >> 4, ap = i >> 1, co = i & 1;
  float mx = 0.f;
  if (t < a.n_tiles) {  // uniform per wave
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      const size_t at = (size_t)t * 256 + 64 * q + lane;
      const float2 x = slot_weight(a.wf, a.w0, a.w1, a.perm[at]);
      a.wc[at] = x;
      s_w[wv][64 * q + lane] = x;
      mx = fmaxf(mx, fmaxf(fabsf(x.x), fabsf(x.y)));
    }
  }
  for (int off = 32; off; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  if (lane == 0) s_max[wv] = mx;
  __syncthreads();
  if (t >= a.n_tiles) return;
  // the workgroup's four tiles hold whole groups (a.n_tiles is a multiple of a.group)
  for (uint32_t o = 0; o < a.group; ++o) mx = fmaxf(mx, s_max[(wv & ~(a.group - 1u)) + o]);
  int e = 0;
  if (mx > 0.f && __builtin_isfinite(mx)) frexpf(mx, &e);
  e = e < -126 ? -126 : (e > 127 ? 127 : e);
  const float is = ldexpf(1.f, -e);
  float2 w[2][4];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int q = 0; q < 4; ++q) w[rb][q] = s_w[wv][16 * (8 * rb + ap) + 4 * g + q];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const float kr = (float)(8 * rb + ap) - 7.5f;
    const float ka = kr * kCrossW, ka2 = kr * kr * kCross2W;
    h8v hi, lo, cr, crl, c2;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float vr = w[rb][q].x * is, vi = w[rb][q].y * is;
      // real form: rows (a, re) = (Vr, -Vi), (a, im) = (Vi, Vr)
      const float A0 = co ? vi : vr, A1 = co ? vr : -vi;
      // i k W: real part -k Wi, imaginary part k Wr
      const float C0 = co ? ka * vr : -ka * vi, C1 = co ? -ka * vi : -ka * vr;
      _Float16 h, l;
      split_f16(A0, h, l);
      hi[2 * q] = h;
      lo[2 * q] = l;
      split_f16(A1, h, l);
      hi[2 * q + 1] = h;
      lo[2 * q + 1] = l;
      split_f16(C0, h, l);
      cr[2 * q] = h;
      crl[2 * q] = l;
      split_f16(C1, h, l);
      cr[2 * q + 1] = h;
      crl[2 * q + 1] = l;
      // k^2 W (real scaling): the same real form as W
      c2[2 * q] = (_Float16)(ka2 * A0);
      c2[2 * q + 1] = (_Float16)(ka2 * A1);
    }
    a.wq[((size_t)t * 6 + 3 * rb + 0) * 64 + lane] = __builtin_bit_cast(uint4, hi);
    a.wq[((size_t)t * 6 + 3 * rb + 1) * 64 + lane] = __builtin_bit_cast(uint4, lo);
    a.wq[((size_t)t * 6 + 3 * rb + 2) * 64 + lane] = __builtin_bit_cast(uint4, cr);
    if (a.wqn) {
      a.wqn[((size_t)t * 4 + 2 * rb + 0) * 64 + lane] = __builtin_bit_cast(uint4, crl);
      a.wqn[((size_t)t * 4 + 2 * rb + 1) * 64 + lane] = __builtin_bit_cast(uint4, c2);
    }
  }
  if (lane == 0) a.tscale[t] = ldexpf(1.f, e);
}

}  // namespace holo
