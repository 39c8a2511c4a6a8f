// Device code shared by the kernels for targets on a uniform lattice
// (holo_pairs.hip, holo_points.hip): the targets' lattice, f16 pair arithmetic on
// the matrix cores, phases as fractions of a cycle.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "holo_device.hpp"
#include "holo_internal.hpp"

namespace holo {

typedef float pf16 __attribute__((ext_vector_type(16)));
typedef _Float16 ph2 __attribute__((ext_vector_type(2)));
typedef _Float16 ph8 __attribute__((ext_vector_type(8)));
typedef uint32_t pu4 __attribute__((ext_vector_type(4)));

// PairTargets::mode: a form, or (lattice to lattice) kPairNear, which holds for every
// tile pair, with kPairWide for the source tiles of 64 columns
constexpr uint32_t kPairFar = 1, kPairNear = 2, kPairWide = 4;
constexpr float kPairMid = 15.5f;  // a 32 x 32 tile's centre
constexpr uint32_t kPairMaxRow = 16384;  // longest row of targets looked for
constexpr int kPairWaves = kBlock / 64;
// Two workgroups of four waves run on a CU (their LDS and VGPRs).
constexpr size_t kPairSlots = 2 * 256;
constexpr float kFourPi = 12.566370614359172f;

// The dropped terms of a tile pair at their largest: rx, ry the lateral distances
// between the tile centres (or the largest of several pairs), hx, hy the largest
// |rho|, id = 1 / D (or of the smallest D).  cross = |C| of the first order.
struct PairTerms {
  bool in_range;
  float cross, cubic, cube, sq, q4;
};

__device__ __forceinline__ PairTerms pair_terms(float rx, float ry, float hx, float hy, float id,
                                                float inv_lambda) {
  // P, Q over D^2, and D / lambda: the same at every scale of lengths
  const float id2 = id * id, dl = inv_lambda / id;
  const float p = (2.f * rx * hx + hx * hx) * id2, q = (2.f * ry * hy + hy * hy) * id2;
  const float big = fmaxf(p, q), sum = p + q;
  PairTerms t;
  // alpha P, which cycles32 has to hold, and c2 P^2, in 2^-32 cycles an int32; w^2, which
  // p is scaled by, is no denormal
  t.in_range = 0.5f * dl * sum <= 0x1p17f && 0.125f * dl * big * big <= 0.25f &&
               id * inv_lambda * id2 >= 0x1p-100f;
  t.cross = 1.5707964f * dl * p * q;
  t.cubic = 1.1780972f * dl * p * q * sum;  // rad, the c3 part of C
  t.cube = 0.0625f * dl * big * big * big;
  t.sq = sum;
  t.q4 = 0.0390625f * dl * sum * sum * sum * sum;
  return t;
}

// Whether the forms hold with cross up to `most`.  NaN gives false.
__device__ __forceinline__ bool pair_far(const PairTerms& t, bool obl, float most) {
  return t.in_range && t.cross <= most && t.cubic <= 1e-6f && t.cube <= 1e-8f &&
         (obl ? 1.f : 0.5f) * t.sq * t.sq <= 1e-7f;
}

__device__ __forceinline__ bool pair_near(const PairTerms& t, float most) {
  return t.in_range && t.cross <= most && t.cubic <= 4e-4f && t.q4 <= 1e-8f &&
         t.sq * t.sq * t.sq <= 1e-7f;
}

// first k in [1, lim) for which hit(k) holds, else lim; the whole workgroup
template <typename F>
__device__ uint32_t block_first(uint32_t lim, uint32_t* s_min, F&& hit) {
  constexpr int kEach = 4;
  for (uint32_t base = 1; base < lim; base += kEach * kBlock) {
    uint32_t first = lim;
#pragma unroll
    for (int q = 0; q < kEach; ++q) {
      const uint32_t k = base + q * kBlock + threadIdx.x;
      if (k < lim && hit(k)) first = min(first, k);
    }
    for (int off = 32; off; off >>= 1)
      first = min(first, (uint32_t)__shfl_xor((int)first, off, 64));
    __syncthreads();  // the previous round's reads of s_min are done
    if ((threadIdx.x & 63) == 0) s_min[threadIdx.x >> 6] = first;
    __syncthreads();
    first = min(min(s_min[0], s_min[1]), min(s_min[2], s_min[3]));
    if (first < lim) return first;
  }
  return lim;
}

// Looks for the targets' lattice: every probe workgroup finds the row length (the
// first target with another x) and the number of rows (the first row that starts
// with target 0's x again: the generator fills up with copies of point 0), then
// checks its share of the targets against x_0 + i p_x, y_0 + j p_y, z_0 to 1e-9 of
// a pitch (a product of one x per row and one y per column to the bit), and the
// rest against target 0.  flags[b] = 1 when its share passes, and `ok` (the caller's
// checks) holds on every lane; workgroup 0 writes
// *pt, with the mode that form(pt, cx0, cx1, cy0, cy1) gives for the lattice of 32 x
// 32 tiles with the first and last centres (cx0, cy0), (cx1, cy1).
template <typename F>
__device__ void probe_targets(const double* __restrict__ v, uint32_t M, uint32_t b,
                              uint32_t n_probe, PairTargets* pt, uint32_t* flags, uint32_t* s_min,
                              bool ok, F&& form) {
  const double x0 = v[0], y0 = v[1], z0 = v[2];
  const uint32_t lim = min(M, kPairMaxRow);
  const uint32_t ny = block_first(lim, s_min, [&](uint32_t k) { return v[3 * (size_t)k] != x0; });
  uint32_t nx = ny < lim && ny >= 16 ? M / ny : 0u;
  if (nx >= 16)
    nx = block_first(nx, s_min, [&](uint32_t k) { return v[3 * (size_t)k * ny] == x0; });
  double px = 0.0, py = 0.0;
  if (nx < 16) {
    ok = false;
  } else {
    const uint32_t body = nx * ny;
    px = (v[3 * (size_t)(nx - 1) * ny] - x0) / (double)(nx - 1);
    py = (v[3 * (size_t)(ny - 1) + 1] - y0) / (double)(ny - 1);
    const double tx = 1e-9 * fabs(px), ty = 1e-9 * fabs(py);
    ok = ok && tx > 0.0 && ty > 0.0 && __builtin_isfinite(px) && __builtin_isfinite(py);
    for (uint32_t m = b * kBlock + threadIdx.x; m < M; m += n_probe * kBlock) {
      const double x = v[3 * (size_t)m], y = v[3 * (size_t)m + 1], z = v[3 * (size_t)m + 2];
      if (m < body) {
        const uint32_t i = m / ny, j = m - i * ny;
        ok = ok && x == v[3 * (size_t)i * ny] && y == v[3 * (size_t)j + 1] && z == z0 &&
             fabs(x - (x0 + (double)i * px)) <= tx && fabs(y - (y0 + (double)j * py)) <= ty;
      } else {
        ok = ok && x == x0 && y == y0 && z == z0;
      }
    }
  }
  const int all = __syncthreads_and(ok ? 1 : 0);
  if (threadIdx.x) return;
  flags[b] = all ? 1u : 0u;
  if (b) return;
  PairTargets t;
  t.x0 = x0;
  t.y0 = y0;
  t.z = z0;
  t.px = px;
  t.py = py;
  t.nx = nx;
  t.ny = ny;
  t.mode = 0u;
  if (all) {
    // tile centres of the targets: first and last
    const double cx0 = x0 + (double)kPairMid * px, cy0 = y0 + (double)kPairMid * py;
    const double cx1 = cx0 + (double)(((nx + 31) / 32 - 1) * 32) * px;
    const double cy1 = cy0 + (double)(((ny + 31) / 32 - 1) * 32) * py;
    t.mode = form(t, cx0, cx1, cy0, cy1);
  }
  *pt = t;
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x added to this lane's own word of LDS, without reading it back
__device__ __forceinline__ void lds_add(double* p, double x) {
  __hip_atomic_fetch_add(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ double lane_f64(double x, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ float lane_f32(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// x + kCycles32 has ulp 2^-32 for |x| < 2^19 - 1: its low word is x modulo one
// cycle, in 2^-32 cycles.
constexpr double kCycles32 = 0x1.8p20;
__device__ __forceinline__ uint32_t cycles32(double x) {
  return (uint32_t)__builtin_bit_cast(uint64_t, x);
}

__device__ __forceinline__ pf16 mfma32(ph8 a, ph8 b, pf16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ ph8 neg8(ph8 x) {
  pu4 u = __builtin_bit_cast(pu4, x);
  u ^= 0x80008000u;
  return __builtin_bit_cast(ph8, u);
}

// (a, b) rounded to nearest f16
typedef float pf2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ ph2 pk(float a, float b) {
  return __builtin_convertvector((pf2{a, b}), ph2);
}

// A product that is split into hi and lo: kept apart from the conversions, as
// the compiler could fold it into the one that gives the operand hi and not into
// the one that lo = x - hi is formed with, and at ties hi + lo would then be off
// by an f16 ulp of x.
__device__ __forceinline__ float formed(float x) {
  __asm__("" : "+v"(x));
  return x;
}

// hi = (x rounded), lo = am x - hi, of eight values (x formed: no product)
__device__ __forceinline__ void split8(const float (&x)[8], const float (&am)[8], ph8& hi,
                                       ph8& lo) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const ph2 t = pk(x[e], x[e + 1]);
    hi[e] = t[0];
    hi[e + 1] = t[1];
    const ph2 d = pk(__builtin_fmaf(am[e], x[e], -(float)t[0]),
                     __builtin_fmaf(am[e + 1], x[e + 1], -(float)t[1]));
    lo[e] = d[0];
    lo[e + 1] = d[1];
  }
}

__device__ __forceinline__ void split8(const float (&x)[8], float one, ph8& hi, ph8& lo) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const ph2 t = pk(x[e], x[e + 1]);
    hi[e] = t[0];
    hi[e + 1] = t[1];
    const ph2 d = pk(__builtin_fmaf(x[e], one, -(float)t[0]),
                     __builtin_fmaf(x[e + 1], one, -(float)t[1]));
    lo[e] = d[0];
    lo[e + 1] = d[1];
  }
}

__device__ __forceinline__ ph8 half8(const float (&x)[8]) {
  ph8 r;
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const ph2 t = pk(x[e], x[e + 1]);
    r[e] = t[0];
    r[e + 1] = t[1];
  }
  return r;
}

// eight values as f16
__device__ __forceinline__ ph8 mul8(ph8 a, ph8 b) { return a * b; }

// (Dr, Di) += complex product of the hi parts of A and B
struct Cplx8 {
  ph8 rh, rl, ih, il;
};

__device__ __forceinline__ void cmul_hi(const Cplx8& a, const Cplx8& b, pf16& Dr, pf16& Di) {
  Dr = mfma32(a.rh, b.rh, Dr);
  Di = mfma32(a.rh, b.ih, Di);
  Dr = mfma32(a.ih, neg8(b.ih), Dr);
  Di = mfma32(a.ih, b.rh, Di);
}

// of hi by lo parts
__device__ __forceinline__ void cmul_hl(const Cplx8& a, const Cplx8& b, pf16& Dr, pf16& Di) {
  Dr = mfma32(a.rh, b.rl, Dr);
  Di = mfma32(a.rh, b.il, Di);
  Dr = mfma32(a.ih, neg8(b.il), Dr);
  Di = mfma32(a.ih, b.rl, Di);
}

// and of hi by lo and lo by hi parts
__device__ __forceinline__ void cmul_lo(const Cplx8& a, const Cplx8& b, pf16& Dr, pf16& Di) {
  cmul_hl(a, b, Dr, Di);
  Dr = mfma32(a.rl, b.rh, Dr);
  Di = mfma32(a.rl, b.ih, Di);
  Dr = mfma32(a.il, neg8(b.ih), Dr);
  Di = mfma32(a.il, b.rh, Di);
}

constexpr pf16 kZero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                          0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

}  // namespace holo
