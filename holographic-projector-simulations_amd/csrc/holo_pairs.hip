// Lattice-to-lattice kernel: FP32-split superposition from sources on a uniform
// lattice to targets on a uniform lattice (planes of the reference's
// generators on both sides, cuda/init.h:89-158), 32 x 64 sources by 32 x 32
// targets at a time as two chained complex GEMMs on the matrix cores.
//
// For a tile of sources (centre c) and a tile of targets (centre t), r = t - c
// and D = |r|, the source at offset delta and the target at offset tau have
//   d^2 = D^2 + P + Q,   P = rho_x^2 + 2 r_x rho_x,  Q = rho_y^2 + 2 r_y rho_y,
//   rho = tau - delta,
// so P depends on the two x offsets only and Q on the two y offsets only, and
//   e^{i s 2 pi d / lambda} / d = A e^{i s 2 pi f} X Y e^{i C},   f = frac(D / lambda)
//   X = (1 + k1 P + ..) e^{i s 2 pi (alpha P + c2 P^2 + ..)},  Y likewise in Q,
//   C = s 2 pi (2 c2 P Q + 3 c3 (P^2 Q + P Q^2) + ..),
//   alpha = 1 / (2 D lambda), c2 = -alpha / (4 D^2), c3 = alpha / (8 D^4).
// With p = w P, w^2 = |c2|, and q = 4 pi w Q, e^{iC} is a short sum of products
// p^j g_j(q), and a tile contributes the matrix products
//   S = sum_j (p^j X) W (g_j Y)^T,   T_j = W (g_j Y)^T first, then (p^j X) T_j:
// 96 x 32 phasors and 96 x 32^2 complex multiply-adds per product for the 2 x 32^4
// pairs of a tile of sources and one of targets.
//   far (rank 2):  g_0 = 1, g_1 = i sigma q,  sigma = -s
//   near (rank 4): g_1 = q (k11 + i (sigma + gQ q)),
//                  g_2 = q (i gP - q / 2 - sigma gQ q^2),
//                  g_3 = -q^2 (sigma gP + i sigma q / 6),
//     gP = s 6 pi c3 / (4 pi w^3), gQ = gP / (4 pi), k11 the amplitude's cross
//     term, and the rows and columns carry c3 P^3 and the quadratic amplitude.
// Every tile pair takes the far form within its bounds and the near form elsewhere.
// Where the bounds ask for it the source tiles are 32 x 32 (halves of the others).
// k_pair_prep picks the width from the near form's bounds over all tile pairs
// (pair_mode), or neither, and then the 16-row kernels run as if this kernel did not
// exist.  (One form for a whole call, far up to cross = 2.4e-3 and near up to 0.12, left
// up to 2.8e-6 of the field for one lit source in a tile's corner; now 5.8e-7.)
//
// Operands are f16 pairs x = hi + lo (both rounded to nearest), and a full
// product is hi hi + hi lo + lo hi, in FP32: only lo lo (2^-22, of either sign)
// is left out.  g_0 and the near form's g_1 are full products; the far form's g_1
// (below 1e-3 of the sum), g_2 (below 4.5e-4, full above) and g_3 (below 1.7e-4) take the
// phasors' and weights' hi parts and both of T's, which are sums (T's hi parts alone:
// 3 to 4 % less time).  X carries A over the planes' 1 / |dz|.  The matrix cores' FP32 sums are rounded to
// one side: in T that is turned by X's phases, but in the second product it would
// add up over the tiles (1.6e-7 of the field over 1024 tiles; 5e-7 when one
// accumulator ran over 16 tiles).  So each tile's products start from zero, every
// other tile with the opposite sign, and are added in FP64; the far form, which
// has the registers for it, keeps the small parts in accumulators of their own.
// Relative L2 against FP64: 1.9e-7 (far), 2.1e-7 (near) at 1024^2 sources; the
// 16-row kernels are at 2.7e-7 to 3.3e-7.
//
// Phases: alpha P = alpha (tau^2 + 2 r_x tau) + alpha (delta^2 - 2 r_x delta) -
// 2 alpha tau delta.  The first two span many cycles over a tile; one lane forms
// each of the 2 x 64 of them in FP64 per tile pair.  They are added, with the
// bilinear part and c2 P^2, as 32-bit fractions of a cycle (exact, and modulo one
// cycle for free), and only the sum, in [-1/2, 1/2), is rounded to FP32.
//
// Layout (v_mfma_f32_32x32x16_f16): lane l = 32 h + j holds eight k of row j of
// A and of column j of B; result register r is row 8 (r / 4) + 4 h + r % 4 of
// column j.  With the k slots of a step s taken as 16 s + 8 (e / 4) + 4 h + e % 4,
// the eight registers 8 s .. 8 s + 7 of T are, without any exchange between
// lanes, the B operand of the second product, and each lane forms its own
// phasors: X of target row j and Y of target column j.  Real and imaginary
// parts are separate operands: T_re = Wr Yr + Wi (-Yi), T_im = Wr Yi + Wi Yr.
//
// What bounds it: VALU issue, 76 % busy (805 instructions per 2^20 pairs at 1024^2 and
// 0.35 m, half of them for the phasors), beside matrix cores at 38 %; two waves per SIMD
// (253 VGPRs).  Per call, 1024^2 -> 1024^2 at 0.35 m: 2.31 to 2.38 ms, 3 % of the tile
// pairs near (one form for all: 2.03 to 2.09 ms), where the 16 x 64 tiles of
// k_superpose_grid16 take 57.8 ms; 3.9 ms at 0.2 m (93 ms; one form 4.5 ms), 6.2 ms at
// 0.1 m (140 ms); 512^2 -> 512^2 at 0.1 m 0.31 ms, 75 % near (8.2 ms); 64^2 -> 64^2: 25
// to 29 us (34 us).  With 32 x 32 source tiles the far form took 1.35 times as long.
#include <hip/hip_runtime.h>
#include <math.h>

#include "holo_device.hpp"
#include "holo_internal.hpp"
#include "holo_mfma.hpp"
#include "holo_weights.hpp"

namespace holo {

constexpr int kPairTile = 32;  // rows and columns of a target tile, rows of a source tile
// MFMA operands of one 32 x 64 source tile's weights by four workgroups, and the
// target lattice by the n_probe workgroups after them (tail sources' weights by
// one before those); the rest, if any, prepare the 16-row kernels' weights.  What bounds
// it is the FP64 sin and cos that a lane forms one after the other: with eight in each
// (one workgroup a tile) a call of 16^2 or 64^2 sources spent 6.6 or 7.5 us here, 5.2 and 4.8 now.
//
// Weights: wq[(16 t + 4 s + 2 c + l) * 64 + lane] (8 f16) holds, for step s < 4
// (columns 16 s ..), component c (re, im) and part l (hi, lo), row delta_x =
// lane % 32 of tile t over its scale tscale[t] (the power of two above its
// largest modulus, or component of complex weights); slots beyond the lattice are 0.
//
// Targets: probe_targets.
struct PairPrep {
  const double* w0;
  const double* w1;
  int wf;
  uint32_t nx, ny, tj, n_tiles, n_tail, tail_same;
  pu4* wq;
  float* tscale;
  float2* tail_wc;
  const double* v;
  uint32_t M, n_probe, obl;
  double sx, sy, sz, spx, spy, inv_lambda;
  PairTargets* pt;
  uint32_t* flags;
};

// Columns 16 step .. 16 step + 15 of tile t: two sources' weights a lane, laid out
// through LDS (s_w: 32 x 17 float2).
__device__ void pair_tile_weights(const PairPrep& a, uint32_t t, uint32_t step, float* s_max,
                                  float2* s_w) {
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t I = t / a.tj, J = t - I * a.tj;
  const auto source = [&](uint32_t row, uint32_t col) {
    const uint32_t i = kPairTile * I + row, j = 2 * kPairTile * J + col;
    return i < a.nx && j < a.ny ? (int32_t)(i * a.ny + j) : -1;
  };
  // the bound of the whole tile's components: the moduli's (polar) or their own
  float mx = 0.f;
#pragma unroll
  for (uint32_t e = 0; e < 8; ++e) {
    const int32_t n = source(4 * e + wv, lane);
    if (n < 0) continue;
    if (a.wf == kPolar)
      mx = fmaxf(mx, fabsf((float)a.w0[n]));
    else
      mx = fmaxf(mx, fmaxf(fabsf((float)a.w0[2 * (size_t)n]), fabsf((float)a.w0[2 * (size_t)n + 1])));
  }
#pragma unroll
  for (uint32_t e = 0; e < 2; ++e) {
    const uint32_t row = 16 * e + (threadIdx.x >> 4), col = threadIdx.x & 15;
    s_w[17 * row + col] = slot_weight(a.wf, a.w0, a.w1, source(row, 16 * step + col));
  }
  for (int off = 32; off; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  if (lane == 0) s_max[wv] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
  int e2 = 0;
  if (mx > 0.f && __builtin_isfinite(mx)) frexpf(mx, &e2);
  e2 = e2 < -126 ? -126 : (e2 > 127 ? 127 : e2);
  const float is = ldexpf(1.f, -e2);
  // wave 2 c + l: component c, part l
  const float2* w = s_w + 17 * (lane & 31) + 4 * (lane >> 5);
  ph8 op;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float2 x = w[8 * (e >> 2) + (e & 3)];
    const float c = (wv & 2 ? x.y : x.x) * is;
    // 11 significant bits by integer rounding: exact in f16, and lo exact
    const float h = __builtin_bit_cast(
        float, (__builtin_bit_cast(uint32_t, c) + 0x1000u) & 0xffffe000u);
    op[e] = (_Float16)(wv & 1 ? c - h : h);
  }
  a.wq[((size_t)16 * t + 4 * step + wv) * 64 + lane] = __builtin_bit_cast(pu4, op);
  if (step == 0 && threadIdx.x == 0) a.tscale[t] = ldexpf(1.f, e2);
}

// FP32 weights of the sources after the lattice; when they all sit at one
// point, their FP64 sum alone (in a fixed order).
__device__ void pair_tail_weights(const PairPrep& a, double* s_red) {
  const uint32_t body = a.nx * a.ny;
  if (!a.tail_same) {
    for (uint32_t k = threadIdx.x; k < a.n_tail; k += kBlock) a.tail_wc[k] = slot_weight(a.wf, a.w0, a.w1, (int32_t)(body + k));
    return;
  }
  double re = 0.0, im = 0.0;
  for (uint32_t k = threadIdx.x; k < a.n_tail; k += kBlock) {
    const uint32_t n = body + k;
    if (a.wf == kPolar) {
      double sn, cs;
      sincos(a.w1[n], &sn, &cs);
      re += a.w0[n] * cs;
      im += a.w0[n] * sn;
    } else {
      re += a.w0[2 * (size_t)n];
      im += a.w0[2 * (size_t)n + 1];
    }
  }
  s_red[threadIdx.x] = re;
  s_red[kBlock + threadIdx.x] = im;
  __syncthreads();
  for (int h = kBlock / 2; h; h >>= 1) {
    if ((int)threadIdx.x < h) {
      s_red[threadIdx.x] += s_red[threadIdx.x + h];
      s_red[kBlock + threadIdx.x] += s_red[kBlock + threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) a.tail_wc[0] = make_float2((float)s_red[0], (float)s_red[kBlock]);
}

// The largest cross a tile pair takes each form with.  The far form drops C^2 / 2 and
// the near form C^4 / 24; with m the pair's largest |C|, lowering the constant to 1 -
// m^2 / 4 leaves at most m^2 / 4 of the one (2.5e-7), and 1 - m^4 / 192 with 1 / 2 -
// m^2 / 24 in the C^2 term at most m^4 / 192 of the other (5.2e-7).  These hold for one lit
// source in the worst corner of its tile; over dense weights C's triangular
// distribution leaves a tenth.  f16 hi parts leave about 2^-12 of a product: of C in the
// far form (2.4e-7), of C^2 / 2 in the near form up to kCrossHi (1.1e-7; full products from
// there on) and of C^3 / 6 above (4e-8).
constexpr float kCrossFar = 1e-3f, kCrossHi = 0.03f, kCrossNear = 0.1f;

// The source tile width for targets with the first and last tile centres (cx0, cy0),
// (cx1, cy1): the wide tiles where the near form holds for every pair of them, but the
// narrow ones where those are all far and the wide ones mostly are not (judged midway
// between the lattices).
__device__ uint32_t pair_mode(const PairPrep& a, const PairTargets& t, double cx0, double cx1,
                              double cy0, double cy1) {
  const auto far = [](double a0, double a1, double b0, double b1) {
    return fmax(fmax(fabs(a0 - b0), fabs(a0 - b1)), fmax(fabs(a1 - b0), fabs(a1 - b1)));
  };
  const auto mid = [](double a0, double a1, double b0, double b1) {
    return 0.5 * fabs(a0 + a1 - b0 - b1);
  };
  // source tile centres: rows, and columns of wide and of narrow tiles
  const double sx0 = a.sx + (double)kPairMid * a.spx;
  const double sx1 = sx0 + (double)(((a.nx + 31) / 32 - 1) * 32) * a.spx;
  const float hx = (float)((double)kPairMid * (fabs(t.px) + fabs(a.spx)));
  const double dz = fabs(t.z - a.sz);
  const float il = (float)a.inv_lambda;
  bool near[2], all_far[2], mid_far[2];
  for (int wide = 0; wide < 2; ++wide) {
    const double half = wide ? 31.5 : (double)kPairMid;
    const uint32_t cols = wide ? 64 : 32;
    const double sy0 = a.sy + half * a.spy;
    const double sy1 = sy0 + (double)(((a.ny + cols - 1) / cols - 1) * cols) * a.spy;
    const float hy = (float)((double)kPairMid * fabs(t.py) + half * fabs(a.spy));
    const PairTerms d = pair_terms((float)far(cx0, cx1, sx0, sx1), (float)far(cy0, cy1, sy0, sy1),
                                   hx, hy, 1.f / (float)dz, il);
    near[wide] = pair_near(d, kCrossNear);
    all_far[wide] = pair_far(d, a.obl != 0, kCrossFar);
    const double mx = mid(cx0, cx1, sx0, sx1), my = mid(cy0, cy1, sy0, sy1);
    mid_far[wide] = pair_far(pair_terms((float)mx, (float)my, hx, hy,
                                        1.f / (float)sqrt(mx * mx + my * my + dz * dz), il),
                             a.obl != 0, kCrossFar);
  }
  if (near[1] && (mid_far[1] || !all_far[0])) return kPairNear | kPairWide;
  return near[0] ? kPairNear : 0u;
}

__global__ __launch_bounds__(kBlock) void k_pair_prep(PairPrep a, Grid16Prep g) {
  __shared__ double s_buf[2 * kBlock + 64];
  static_assert(sizeof(s_buf) >= 32 * 17 * sizeof(float2) + kPairWaves * sizeof(float), "s_w, s_max");
  uint32_t b = blockIdx.x;
  if (b < 4 * a.n_tiles) {
    float2* s_w = reinterpret_cast<float2*>(s_buf);
    pair_tile_weights(a, b >> 2, b & 3, reinterpret_cast<float*>(s_w + 32 * 17), s_w);
    return;
  }
  b -= 4 * a.n_tiles;
  if (a.n_tail) {
    if (b == 0) {
      pair_tail_weights(a, s_buf);
      return;
    }
    --b;
  }
  if (b < a.n_probe)
    probe_targets(a.v, a.M, b, a.n_probe, a.pt, a.flags, reinterpret_cast<uint32_t*>(s_buf), true,
                  [&](const PairTargets& t, double cx0, double cx1, double cy0, double cy1) {
                    return pair_mode(a, t, cx0, cx1, cy0, cy1);
                  });
  else
    grid16_weights(g, b - a.n_probe);
}

// One wave's LDS: FP64 sums of its target tile, and the tile pair's fractions
// and offsets per row and column: phase fractions and parts of p (q) of the
// targets (entry 32 axis + index) and of the sources (rows at 0, columns at 32).
struct PairLds {
  double re[kPairWaves][16][64];
  double im[kPairWaves][16][64];
  uint32_t tF[kPairWaves][64], sF[kPairWaves][96];
  float tp[kPairWaves][64], sp[kPairWaves][96];
};

// Eight phasors of one step: (c, s), their p (or q) and amplitude.
struct Phasors {
  float c[8], s[8], p[8], am[8];
};

// ---- one wave, one target tile, the source tiles of one split ----
template <int SIGN, bool OBL>
struct PairWave {
  PairLds& lds;
  uint32_t lane, wv, h, j;
  // per tile pair
  uint32_t FtX, FtY;          // phase of this lane's row, column and source slot 0 (2^-32 cycles)
  float PtX, PtY;             // and its part of p, q
  uint32_t cbX, cbY;          // bilinear coefficients per source index
  float pbX, pbY;
  float a0X, a1X, a2X;        // X's amplitude in p: A |dz| (1 + k1 P + k2 P^2)
  float a1Y, a2Y;             // Y's: 1 + k1 Q + k2 Q^2
  float c3X, c3Y, k11, gP, gQ;  // near form (c3X, c3Y in 2^-32 cycles)
  float half;                   // near form: the C^2 term's coefficient
  float one;                  // 1, unknown to the compiler: x - hi as one mixed FMA

  // phasors of step s along AXIS (0: x, 1: y)
  template <bool NEAR, int AXIS>
  __device__ __forceinline__ void phasors(uint32_t s, Phasors& o) const {
    const uint32_t cb = AXIS ? cbY : cbX, F = (AXIS ? FtY : FtX) + 16u * s * cb;
    const float pb = AXIS ? pbY : pbX, P0 = __builtin_fmaf(pb, (float)(16 * s), AXIS ? PtY : PtX);
    // c2 P^2 = -p^2, c2 Q^2 = -(q / 4 pi)^2, in 2^-32 cycles
    constexpr float kC2 = (AXIS ? -0.006332573977646111f : -1.f) * 0x1p32f;
    const float a1 = AXIS ? a1Y : a1X, a2 = AXIS ? a2Y : a2X, c3 = AXIS ? c3Y : c3X;
    const float a0 = AXIS ? 1.f : a0X;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint32_t at = 32 * AXIS + 16 * s + 8 * q + 4 * h;
      const uint4 f4 = *reinterpret_cast<const uint4*>(&lds.sF[wv][at]);
      const float4 p4 = *reinterpret_cast<const float4*>(&lds.sp[wv][at]);
      const uint32_t fs[4] = {f4.x, f4.y, f4.z, f4.w};
      const float ps[4] = {p4.x, p4.y, p4.z, p4.w};
      const uint32_t Fq = F + cb * (uint32_t)(8 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p = __builtin_fmaf(pb, (float)(8 * q + e), P0 + ps[e]);
        const float pp = p * p;
        const int32_t t2 = (int32_t)(pp * (NEAR ? __builtin_fmaf(c3, p, kC2) : kC2));
        const float t =
            (float)(int32_t)(Fq + cb * (uint32_t)e + fs[e] + (uint32_t)t2) * 0x1p-32f;
        float sn, cs;
        sincos_rev_f32(t, sn, cs);
        o.c[4 * q + e] = cs;
        o.s[4 * q + e] = SIGN > 0 ? sn : -sn;
        o.p[4 * q + e] = p;
        o.am[4 * q + e] = __builtin_fmaf(p, NEAR ? __builtin_fmaf(a2, p, a1) : a1, a0);
      }
    }
  }
};

// registers 8 s .. 8 s + 7 of T as the second product's B operand
__device__ __forceinline__ Cplx8 operand_of(const pf16& Tr, const pf16& Ti, int s, float one) {
  Cplx8 o;
  float r[8], i[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    r[e] = Tr[8 * s + e];
    i[e] = Ti[8 * s + e];
  }
  split8(r, one, o.rh, o.rl);
  split8(i, one, o.ih, o.il);
  return o;
}

// PART 0: the far form (g_0 full, g_1 hi parts); PART 1, 2: the near form's g_0,
// g_1 (full) and g_2, g_3 (hi parts); PART 3: as 2 with g_2 full.  Adds the products of a tile with `steps`
// steps of 16 columns (weights wt) into (Dr, Di).
template <int PART, int SIGN, bool OBL>
__device__ __forceinline__ void pair_products(const PairWave<SIGN, OBL>& pw, const pu4* wt,
                                              uint32_t steps, pf16& Dr, pf16& Di) {
  constexpr bool NEAR = PART != 0, FULL_A = PART == 1 || PART == 3;
  constexpr float kSig = SIGN > 0 ? -1.f : 1.f;
  pf16 Ar = kZero16, Ai = kZero16, Br = kZero16, Bi = kZero16;
  pf16 Lr = kZero16, Li = kZero16;  // far form: the small parts, apart
#pragma unroll 1
  for (uint32_t s = 0; s < steps; ++s) {
    Cplx8 w;
    w.rh = __builtin_bit_cast(ph8, wt[(4 * s + 0) * 64 + pw.lane]);
    w.rl = __builtin_bit_cast(ph8, wt[(4 * s + 1) * 64 + pw.lane]);
    w.ih = __builtin_bit_cast(ph8, wt[(4 * s + 2) * 64 + pw.lane]);
    w.il = __builtin_bit_cast(ph8, wt[(4 * s + 3) * 64 + pw.lane]);
    Phasors y;
    pw.template phasors<NEAR, 1>(s, y);
    Cplx8 a, b;
    if constexpr (PART == 0) {
      split8(y.c, y.am, a.rh, a.rl);
      split8(y.s, y.am, a.ih, a.il);
      // i sigma q (c + i s)
      const ph8 q = half8(y.p);
      b.rh = mul8(SIGN > 0 ? q : neg8(q), a.ih);
      b.ih = mul8(SIGN > 0 ? neg8(q) : q, a.rh);
      cmul_hi(w, b, Br, Bi);
      cmul_lo(w, a, Lr, Li);
      cmul_hi(w, a, Ar, Ai);
    } else {
      float ar[8], ai[8], br[8], bi[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float q = y.p[e], yr = y.am[e] * y.c[e], yi = y.am[e] * y.s[e];
        float gr, gi;
        if constexpr (PART == 1) {
          gr = pw.k11 * q;
          gi = q * __builtin_fmaf(pw.gQ, q, kSig);
        } else {
          const float q2 = q * q;
          const float hr = -q2 * __builtin_fmaf(kSig * pw.gQ, q, pw.half), hi = pw.gP * q;
          ar[e] = formed(hr * yr - hi * yi);
          ai[e] = formed(hr * yi + hi * yr);
          gr = -kSig * pw.gP * q2;
          gi = (-kSig / 6.f) * (q2 * q);
        }
        br[e] = formed(gr * yr - gi * yi);
        bi[e] = formed(gr * yi + gi * yr);
      }
      if constexpr (PART == 1) {
        split8(br, pw.one, b.rh, b.rl);
        split8(bi, pw.one, b.ih, b.il);
      } else {
        b.rh = half8(br);
        b.ih = half8(bi);
      }
      if constexpr (PART == 1) cmul_lo(w, b, Br, Bi);
      cmul_hi(w, b, Br, Bi);
      __builtin_amdgcn_sched_barrier(0);  // fewer live operands
      if constexpr (PART == 1) {
        split8(y.c, y.am, a.rh, a.rl);
        split8(y.s, y.am, a.ih, a.il);
      } else if constexpr (PART == 3) {
        split8(ar, pw.one, a.rh, a.rl);
        split8(ai, pw.one, a.ih, a.il);
      } else {
        a.rh = half8(ar);
        a.ih = half8(ai);
      }
      if constexpr (FULL_A) cmul_lo(w, a, Ar, Ai);
      cmul_hi(w, a, Ar, Ai);
    }
  }
  if constexpr (PART == 0) {
    Ar += Lr;
    Ai += Li;
    Lr = kZero16;
    Li = kZero16;
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    Phasors x;
    pw.template phasors<NEAR, 0>(s, x);
    Cplx8 a, b;
    float ar[8], ai[8];
    if constexpr (PART == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        ar[e] = formed(x.am[e] * x.c[e]);
        ai[e] = formed(x.am[e] * x.s[e]);
      }
      split8(ar, pw.one, a.rh, a.rl);
      split8(ai, pw.one, a.ih, a.il);
      const ph8 p = half8(x.p);
      b.rh = mul8(p, a.rh);
      b.ih = mul8(p, a.ih);
    } else {
      float br[8], bi[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = x.p[e];
        const float a1 = PART == 1 ? x.am[e] : x.am[e] * (p * p);
        ar[e] = formed(a1 * x.c[e]);
        ai[e] = formed(a1 * x.s[e]);
        br[e] = formed(p * ar[e]);
        bi[e] = formed(p * ai[e]);
      }
      if constexpr (FULL_A) {
        split8(ar, pw.one, a.rh, a.rl);
        split8(ai, pw.one, a.ih, a.il);
      } else {
        a.rh = half8(ar);
        a.ih = half8(ai);
      }
      if constexpr (PART == 1) {
        split8(br, pw.one, b.rh, b.rl);
        split8(bi, pw.one, b.ih, b.il);
      } else {
        b.rh = half8(br);
        b.ih = half8(bi);
      }
    }
    const Cplx8 tb = operand_of(Br, Bi, s, pw.one);
    if constexpr (PART == 0) {
      cmul_hl(b, tb, Lr, Li);
      cmul_hi(b, tb, Lr, Li);
    } else {
      if constexpr (PART == 1) cmul_lo(b, tb, Dr, Di);
      if constexpr (PART >= 2) cmul_hl(b, tb, Dr, Di);
      cmul_hi(b, tb, Dr, Di);
    }
    const Cplx8 ta = operand_of(Ar, Ai, s, pw.one);
    if constexpr (PART == 0) cmul_lo(a, ta, Lr, Li);
    if constexpr (FULL_A) cmul_lo(a, ta, Dr, Di);
    if constexpr (PART == 2) cmul_hl(a, ta, Dr, Di);
    cmul_hi(a, ta, Dr, Di);
  }
  if constexpr (PART == 0) {
    Dr += Lr;
    Di += Li;
  }
}

struct PairSources {
  const pu4* wq;
  const float* tscale;
  double x0, y0, z, px, py;
  uint32_t ny, tj, n_tiles;  // 32 x 64 tiles, tj per row of tiles
  const double* u;
  const int32_t* tail_perm;
  const float2* tail_wc;
  uint32_t n_tail;  // entries of tail_wc
};

// The items of one workgroup: item = target tile x split of the source tiles,
// workgroup b takes items b, b + gridDim.x, ...  The split's source tiles are
// shared out over the workgroup's waves, whose sums are added at the end, so that
// a call of few tiles still occupies four SIMDs a tile and most calls have one
// split, which writes the result itself.
template <int SIGN, bool OBL>
__device__ __forceinline__ void pair_items(PairWave<SIGN, OBL>& pw, const PairSources& sr,
                                           const PairTargets& pt, uint32_t S, uint32_t M,
                                           double inv_lambda, double2* __restrict__ out) {
  PairLds& lds = pw.lds;
  const uint32_t lane = pw.lane, wv = pw.wv, h = pw.h, j = pw.j;
  const uint32_t TI = (pt.nx + 31) / 32, TJ = (pt.ny + 31) / 32, T = TI * TJ;
  const uint32_t items = T * S, parts = kPairWaves * S;
  // this lane's offsets along axis h (FP64), and along both axes (FP32)
  const double ti = (double)j - (double)kPairMid;
  // wide tiles where every wave gets one (else narrow ones, whose bounds are
  // looser: they share the work of a small call better)
  const bool wide = (pt.mode & kPairWide) != 0 && sr.n_tiles >= parts;
  const double midY = wide ? 31.5 : (double)kPairMid;  // the column centre of a source tile
  const double tau = ti * (h ? pt.py : pt.px);
  const double del = h ? ((double)j - midY) * sr.py : ti * sr.px;
  const double del3 = ((double)(32 + j) - midY) * sr.py;  // columns 32 .. 63 of a wide tile
  // source tiles of this mode, tj per row; a wide tile may lack its second half,
  // whose weights are then 0
  const uint32_t stj = wide ? sr.tj : (sr.ny + 31) / 32;
  const uint32_t nst = sr.n_tiles / sr.tj * stj, chunk = (nst + parts - 1) / parts * kPairWaves;
  const double bX = -2.0 * (ti * pt.px * sr.px), bY = -2.0 * (ti * pt.py * sr.py);
  // slot 0's source, from the centre, along x and y
  const double hKX = 4.0 * (double)h - (double)kPairMid, hKY = 4.0 * (double)h - midY;
  const double rz = pt.z - sr.z;
  const float arz = (float)fabs(rz);
  const double irz = 1.0 / fabs(rz);  // X's amplitude is relative to it
  const float hx = (float)((double)kPairMid * (fabs(pt.px) + fabs(sr.px)));
  const float hy = (float)((double)kPairMid * fabs(pt.py) + midY * fabs(sr.py));
  for (uint32_t item = blockIdx.x; item < items; item += gridDim.x) {
    const uint32_t split = item % S, tile = item / S;
    const uint32_t I = tile / TJ, J = tile - I * TJ;
    const double tcx = pt.x0 + ((double)(32 * I) + (double)kPairMid) * pt.px;
    const double tcy = pt.y0 + ((double)(32 * J) + (double)kPairMid) * pt.py;
    // this wave's source tiles: s0 + wv, + 4, .. of the split's (the ones that take the
    // near form lie side by side: with a run of tiles for each wave one wave had them
    // all, and 1024^2 to 1024^2 took 2.5 ms)
    const uint32_t s0 = min(nst, split * chunk), s1 = min(nst, s0 + chunk);
    const uint32_t n = s1 > s0 + wv ? (s1 - s0 - wv + kPairWaves - 1) / kPairWaves : 0u;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      lds.re[wv][r][lane] = 0.0;
      lds.im[wv][r][lane] = 0.0;
    }
    for (uint32_t base = 0; base < n; base += 64) {
      // the FP64 constants of up to 64 source tiles, one per lane
      double hrx, hry, hal, hf;
      float hid, hcr;
      uint64_t far;
      {
        const uint32_t t = s0 + wv + kPairWaves * min(base + lane, n - 1);
        const uint32_t si = t / stj, sj = t - si * stj;
        hrx = tcx - (sr.x0 + ((double)(32 * si) + (double)kPairMid) * sr.px);
        hry = tcy - (sr.y0 + ((double)((wide ? 64 : 32) * sj) + midY) * sr.py);
        double d, id;
        hm_sqrt_inv(__builtin_fma(rz, rz, __builtin_fma(hry, hry, hrx * hrx)), d, id);
        hal = 0.5 * id * inv_lambda;
        hf = frac_cycle(d * inv_lambda);
        hid = (float)id;
        const PairTerms d2 = pair_terms(fabsf((float)hrx), fabsf((float)hry), hx, hy, hid,
                                        (float)inv_lambda);
        hcr = d2.cross;
        far = __builtin_amdgcn_ballot_w64(pair_far(d2, OBL, kCrossFar));
      }
      const uint32_t cnt = min(64u, n - base);
      for (uint32_t k = 0; k < cnt; ++k) {
        const uint32_t t = s0 + wv + kPairWaves * (base + k);
        const double rx = lane_f64(hrx, (int)k), ry = lane_f64(hry, (int)k);
        const double al = lane_f64(hal, (int)k), f = lane_f64(hf, (int)k);
        const float id = lane_f32(hid, (int)k), cross = lane_f32(hcr, (int)k);
        const float id2 = id * id, alf = (float)al;
        // p = w P with w^2 = |c2| = alpha / (4 D^2), q = 4 pi w Q
        const float w = 0.5f * id * __builtin_amdgcn_sqrtf(alf);
        const float iw = __builtin_amdgcn_rcpf(w), wY = kFourPi * w, wA = h ? wY : w;
        {
          const double r2 = 2.0 * (h ? ry : rx);
          const double gt = tau * (tau + r2), gs = del * (del - r2);
          wave_sync();  // the previous tile's reads are done
          lds.tF[wv][lane] = cycles32(__builtin_fma(al, gt, h ? kCycles32 : kCycles32 + f));
          lds.tp[wv][lane] = wA * (float)gt;
          lds.sF[wv][lane] = cycles32(__builtin_fma(al, gs, kCycles32));
          lds.sp[wv][lane] = wA * (float)gs;
          if (wide) {  // uniform
            const double g3 = del3 * (del3 - 2.0 * ry);
            if (!h) {
              lds.sF[wv][64 + j] = cycles32(__builtin_fma(al, g3, kCycles32));
              lds.sp[wv][64 + j] = wY * (float)g3;
            }
          }
          wave_sync();
        }
        // bilinear parts, per source index and at slot 0
        pw.cbX = cycles32(__builtin_fma(al, bX, kCycles32));
        pw.cbY = cycles32(__builtin_fma(al, bY, kCycles32));
        pw.pbX = w * (float)bX;
        pw.pbY = wY * (float)bY;
        pw.FtX = lds.tF[wv][j] + cycles32(__builtin_fma(al, bX * hKX, kCycles32));
        pw.FtY = lds.tF[wv][32 + j] + cycles32(__builtin_fma(al, bY * hKY, kCycles32));
        pw.PtX = __builtin_fmaf(pw.pbX, (float)hKX, lds.tp[wv][j]);
        pw.PtY = __builtin_fmaf(pw.pbY, (float)hKY, lds.tp[wv][32 + j]);
        // the weights: tile t, or for narrow tiles one half of a wide one
        const uint32_t ti2 = wide ? t : (t / stj) * sr.tj + (t % stj) / 2;
        const pu4* wt = sr.wq + (size_t)ti2 * 1024 + (!wide && (t % stj) % 2 ? 512 : 0);
        const uint32_t steps = wide ? 4u : 2u;
        const float tst = sr.tscale[ti2];
        const float iY = (1.f / kFourPi) * iw;  // 1 / wY
        const bool near = !(far >> k & 1);  // uniform
        pw.a0X = OBL ? (arz * id) * (arz * id) : arz * id;
        const float c2 = cross * cross;
        pw.a0X -= (near ? (1.f / 192.f) * c2 * c2 : 0.25f * c2) * pw.a0X;
        pw.a1X = pw.a0X * ((OBL ? -1.f : -0.5f) * id2 * iw);
        pw.a1Y = (OBL ? -1.f : -0.5f) * id2 * iY;
        // every other tile enters the matrix cores with the opposite sign
        pw.FtX += k << 31;
        const float unit = k & 1 ? -tst : tst;
        const auto add = [&](auto part) __attribute__((always_inline)) {
          pf16 Dr = kZero16, Di = kZero16;
          pair_products<decltype(part)::value>(pw, wt, steps, Dr, Di);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            lds_add(&lds.re[wv][r][lane], (double)(unit * Dr[r]));
            lds_add(&lds.im[wv][r][lane], (double)(unit * Di[r]));
          }
        };
        if (!near) {
          add(IC<0>{});
        } else {
          constexpr float k2 = OBL ? 1.f : 0.375f, k11 = OBL ? 1.f : 0.5f;
          pw.a2X = pw.a0X * (k2 * (id2 * iw) * (id2 * iw));
          pw.a2Y = k2 * (id2 * iY) * (id2 * iY);
          // c3 = |c2| id2 / 2:  c3 P^3 = c3X p^3, c3 Q^3 = c3Y q^3
          pw.c3X = 0x1p31f * id2 * iw;
          pw.c3Y = (0x1p31f / (kFourPi * kFourPi)) * id2 * iY;
          pw.k11 = k11 * (id2 * iw) * (id2 * iY);
          pw.gP = (float)SIGN * 9.424778f * id2 * iY;              // s 6 pi c3 / (w^2 wY)
          pw.gQ = (float)SIGN * 9.424778f / kFourPi * id2 * iY;   // s 6 pi c3 / (w wY^2)
          pw.half = __builtin_fmaf(-1.f / 24.f, c2, 0.5f);
          add(IC<1>{});
          // the same phasors again: kept from the first part, and with its results,
          // they would not fit the registers
          __asm__ volatile("" : "+v"(pw.FtX), "+v"(pw.FtY), "+v"(pw.PtX), "+v"(pw.PtY) : : "memory");
          if (cross <= kCrossHi)  // uniform
            add(IC<2>{});
          else
            add(IC<3>{});
        }
      }
    }
    __syncthreads();
    // results: wave v adds up and writes registers 4 v .. 4 v + 3 of the waves' sums,
    // with this split's share of the sources after the lattice
    const uint32_t q0 = (uint32_t)((uint64_t)split * sr.n_tail / S);
    const uint32_t q1 = (uint32_t)((uint64_t)(split + 1) * sr.n_tail / S);
    double2* dst = out + (size_t)split * M;
    const uint32_t col = 32 * J + j;
    for (uint32_t r = 4 * wv; r < 4 * wv + 4; ++r) {
      const uint32_t row = 32 * I + 8 * (r >> 2) + 4 * h + (r & 3);
      double yr = 0.0, yi = 0.0;
#pragma unroll
      for (int k = 0; k < kPairWaves; ++k) {  // fixed order: deterministic
        yr += lds.re[k][r][lane];
        yi += lds.im[k][r][lane];
      }
      yr *= irz;
      yi *= irz;
      if (q1 > q0) {
        const double vx = pt.x0 + (double)row * pt.px, vy = pt.y0 + (double)col * pt.py;
        for (uint32_t q = q0; q < q1; q += 256)
          exact_tile_pairs<SIGN, OBL>(sr.u, sr.tail_perm + q, sr.tail_wc + q,
                                      (int)min(256u, q1 - q), vx, vy, pt.z, inv_lambda, yr, yi);
      }
      if (row < pt.nx && col < pt.ny) dst[(size_t)row * pt.ny + col] = make_double2(yr, yi);
      if (tile == 0 && r == 0) {  // copies of target 0 after the lattice
        const double cr = lane_f64(yr, 0), ci = lane_f64(yi, 0);
        for (uint32_t m = pt.nx * pt.ny + lane; m < M; m += 64) dst[m] = make_double2(cr, ci);
      }
    }
    __syncthreads();  // the sums are read before the next item clears them
  }
}

// handled: 1 when this kernel computes the call, 0 when the 16-row kernels have
// to.
template <int SIGN, bool OBL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, 2))) void
k_superpose_pairs(PairSources sr, const PairTargets* __restrict__ ptp,
                  const uint32_t* __restrict__ flags, uint32_t n_flags, uint32_t* handled,
                  uint32_t S, uint32_t M, double inv_lambda, double2* __restrict__ out) {
  __shared__ PairLds lds;
  const PairTargets pt = *ptp;
  bool good = pt.mode != 0u;
  for (uint32_t k = threadIdx.x; k < n_flags; k += kBlock) good = good && flags[k] != 0u;
  const bool ok = __syncthreads_and(good ? 1 : 0) != 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *handled = ok ? 1u : 0u;
  if (!ok) return;  // uniform
  PairWave<SIGN, OBL> pw{lds, threadIdx.x & 63,
                         (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                         (threadIdx.x & 63) >> 5, threadIdx.x & 31};
  pw.one = 1.f;
  __asm__("" : "+v"(pw.one));
  pair_items<SIGN, OBL>(pw, sr, pt, S, M, inv_lambda, out);
}

// One split where the target tiles fill the slots many times over; else the
// count (at most 8 above one round) that leaves the last round fullest, each
// wave with a source tile of its own.
int pair_splits(size_t M, size_t n_tiles) {
  const Tuning& tu = tuning();
  const size_t most = std::max<size_t>(2 * n_tiles / kPairWaves, 1);
  if (tu.splits > 0) return (int)std::min<size_t>(tu.splits, most);
  // up to four tiles the reduction's launch costs what a second split gives, on either
  // path (56 x 84 sources to 43 x 81 targets: 24.5 us in two splits, 21.8 in one)
  if (most < 3) return 1;
  const size_t tiles = (M + kPairTile * kPairTile - 1) / (kPairTile * kPairTile);
  if (tiles * 8 <= kPairSlots)
    return (int)std::min<size_t>(std::min<size_t>(kPairSlots / tiles, most), 64);
  size_t best = 1;
  double cost = 1e30;
  for (size_t S = 1; S <= std::min<size_t>(most, 8); ++S) {
    const size_t rounds = (tiles * S + kPairSlots - 1) / kPairSlots;
    const double c = (double)rounds / (double)S * (S > 1 ? 1.03 + 0.01 * (double)S : 1.0);
    if (c < cost) {
      cost = c;
      best = S;
    }
  }
  return (int)best;
}

hipError_t launch_superpose_pairs(int sign, bool obliquity, const PairPlan& pp, WeightForm wf,
                                  const double* w0, const double* w1, const double* v, size_t M,
                                  double lambda, int S, PairTargets* pt, uint32_t* flags,
                                  uint32_t* handled, double2* out, const Grid16Prep* grid16,
                                  hipStream_t stream) {
  if (M == 0 || !pp.n_tiles) return hipErrorInvalidValue;
  const uint32_t n_probe = (uint32_t)std::min<size_t>(std::max<size_t>(M / kBlock, 1), kPairFlags);
  PairPrep a;
  a.w0 = w0;
  a.w1 = w1;
  a.wf = (int)wf;
  a.nx = pp.nx;
  a.ny = pp.ny;
  a.tj = pp.tj;
  a.n_tiles = pp.n_tiles;
  a.n_tail = pp.n_tail;
  a.tail_same = pp.tail_same ? 1u : 0u;
  a.wq = reinterpret_cast<pu4*>(pp.wq);
  a.tscale = pp.tscale;
  a.tail_wc = pp.tail_wc;
  a.v = v;
  a.M = (uint32_t)M;
  a.n_probe = n_probe;
  a.obl = obliquity ? 1u : 0u;
  a.sx = pp.x0;
  a.sy = pp.y0;
  a.sz = pp.z;
  a.spx = pp.px;
  a.spy = pp.py;
  a.inv_lambda = 1.0 / lambda;
  a.pt = pt;
  a.flags = flags;
  const Grid16Prep g = grid16 ? *grid16 : Grid16Prep{};
  const unsigned blocks = 4 * pp.n_tiles + (pp.n_tail ? 1u : 0u) + n_probe +
                          (grid16 ? grid16_weight_blocks(g) : 0u);
  k_pair_prep<<<blocks, kBlock, 0, stream>>>(a, g);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  PairSources sr;
  sr.wq = reinterpret_cast<const pu4*>(pp.wq);
  sr.tscale = pp.tscale;
  sr.x0 = pp.x0;
  sr.y0 = pp.y0;
  sr.z = pp.z;
  sr.px = pp.px;
  sr.py = pp.py;
  sr.ny = pp.ny;
  sr.tj = pp.tj;
  sr.n_tiles = pp.n_tiles;
  sr.u = pp.u;
  sr.tail_perm = pp.tail_perm;
  sr.tail_wc = pp.tail_wc;
  sr.n_tail = pp.n_tail ? (pp.tail_same ? 1u : pp.n_tail) : 0u;
  // enough workgroups for every item of a lattice of M targets, at most the
  // resident ones
  const size_t tiles = (M / 1024 + 1) * 4;
  const unsigned grid = (unsigned)std::min<size_t>(tiles * (size_t)S, kPairSlots);
  with_sign(sign, [&](auto sg) {
    with_bool(obliquity, [&](auto obl) {
      k_superpose_pairs<sg.value, (bool)obl.value><<<grid, kBlock, 0, stream>>>(
          sr, pt, flags, n_probe, handled, (uint32_t)S, (uint32_t)M, 1.0 / lambda, out);
    });
  });
  return hipGetLastError();
}

}  // namespace holo
