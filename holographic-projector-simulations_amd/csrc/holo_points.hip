// Point-to-lattice kernel: FP32-split superposition from sources anywhere (the
// reference's jittered pixels and 3-D objects) to targets on a uniform lattice, 16
// sources by 32 x 32 targets at a time as a complex GEMM on the matrix cores.
//
// For a tile of targets (centre t) and a source u_n, r = t - u_n and D = |r| (FP64,
// each source its own), the target at offset tau has d^2 = D^2 + P + Q with
//   P = tau_x^2 + 2 r_x tau_x,   Q = tau_y^2 + 2 r_y tau_y,
// so the expansion of holo_pairs.hip holds with tau in place of tau - delta: with
// its X, Y, p, q and g_j,
//   S[tau_x, tau_y] = sum_n sum_j (w_n A e^{i s 2 pi f} p^j X)[tau_x, n] (g_j Y)[tau_y, n],
// a complex product over the sources, 64 phasors for the 1024 pairs of a source and
// a tile where the tiled kernel (k_superpose_f32s) forms one per pair.  Forms, f16
// pairs and integer phases are those of holo_pairs.hip.  The far form needs
// cross <= 1.2e-3 here: tau is uniform over a tile, so the mean square of cross^2 /
// 2 is 0.2 of its largest, 1.4e-7 furthest off axis (near form: 0.11 cross^4 / 24,
// 1e-7 at 0.07).
//
// Work split: a workgroup takes a tile of targets and its four waves the batches of
// 64 slots (sources in the tiled kernel's order) of one split in turn.  Per batch
// every lane forms one source's FP64 constants and shares them through LDS; per
// step of 16 sources lane 32 h + j forms X of target row j and Y of target column j
// for sources 8 h .. 8 h + 7 of the step, which are its k slots of
// v_mfma_f32_32x32x16_f16's A and B.  A batch's w A are divided by a power of two
// (clouds reach far behind their nearest source).  Its sums start from zero, hi products apart from the small parts, every
// other batch with the opposite sign (the matrix cores round to one side), and are
// added in FP64 in LDS (every second batch: the same time, 1.83e-7 instead of 1.68e-7
// of the field).
//
// What bounds it: VALU issue, 84 % busy (434 instructions per 16 x 1024 pairs, 14 per
// phasor), beside matrix cores at 23 %; two waves per SIMD (238 VGPRs, 79.9 KB of LDS).
// 400^2 jittered sources to 512^2 targets at 0.35 m: 2.46 ms (1.7e13 pairs/s) where
// k_superpose_f32s takes 13.2 ms; near form, 200^2 to 256^2 at 0.05 m: 0.38 and 2.15 ms.
// Relative L2 against FP64 1.7e-7 and 1.9e-7 (2.2e-7 and 4.0e-7).  alpha tau^2 spans
// many cycles on coarse targets and is part of the FP64 phase: as an FP32 addend it
// took the same time and 3.5e-7 at 20 um and 0.05 m (now 1.6e-7).
#include <hip/hip_runtime.h>
#include <math.h>

#include "holo_device.hpp"
#include "holo_internal.hpp"
#include "holo_mfma.hpp"

namespace holo {

constexpr int kPointBatch = 64;  // sources whose constants a wave forms at a time

struct PointLds {
  double re[kPairWaves][16][64];
  double im[kPairWaves][16][64];
  // per source of the batch: linear phases along x and y (cycles per target index);
  // alpha, constant phase + kCycles32; (p and q per target index, k1 / w for Y
  // (near: id2 / w), w); (X's amplitude, the same times k1 / w)
  double2 a1[kPairWaves][kPointBatch];
  double2 f[kPairWaves][kPointBatch];
  float4 p1[kPairWaves][kPointBatch];
  float2 c[kPairWaves][kPointBatch];
};

// Eight phasors (c, s) along AXIS for the sources at 16 s + 8 h .. of the batch, with
// p (or q) and the amplitude.
template <int SIGN, bool OBL>
struct PointWave {
  PointLds& lds;
  uint32_t lane, wv, h, j;
  double kd;            // target index from the tile's centre
  float kf;
  float quad[2];        // (pitch index)^2, per axis: P's quadratic part
  double quad64[2];     // pitch^2 index
  float one;            // 1, unknown to the compiler (split8)

  template <bool NEAR, int AXIS>
  __device__ __forceinline__ void phasors(int s, float (&c)[8], float (&sn)[8], float (&p)[8],
                                          float (&am)[8], float (&g)[8]) const {
    constexpr float kScale = AXIS ? kFourPi : 1.f;  // q = 4 pi w Q
    constexpr float kC2 = (AXIS ? -0.006332573977646111f : -1.f) * 0x1p32f;
    constexpr float kC3 = AXIS ? 0x1p31f / (kFourPi * kFourPi * kFourPi) : 0x1p31f;
    // k2 P^2 = k21 (k1 P)^2
    constexpr float k21 = OBL ? 1.f : 1.5f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t n = 16 * s + 8 * h + e;
      const float4 k = lds.p1[wv][n];
      const double a1 = AXIS ? lds.a1[wv][n].y : lds.a1[wv][n].x;
      const double2 f = lds.f[wv][n];
      p[e] = __builtin_fmaf(k.w, kScale * quad[AXIS], kf * (AXIS ? k.y : k.x));
      const float t2 = p[e] * p[e] * (NEAR ? __builtin_fmaf(kC3 * k.z, p[e], kC2) : kC2);
      const uint32_t t1 = cycles32(
          __builtin_fma(__builtin_fma(f.x, quad64[AXIS], a1), kd, AXIS ? kCycles32 : f.y));
      const float t = (float)(int32_t)(t1 + (uint32_t)(int32_t)t2) * 0x1p-32f;
      float si, co;
      sincos_rev_f32(t, si, co);
      c[e] = co;
      sn[e] = SIGN > 0 ? si : -si;
      g[e] = k.z;
      // 1 + k1 P + k2 P^2, X's times its amplitude
      if constexpr (NEAR) {
        constexpr float k1 = (OBL ? -1.f : -0.5f) / (AXIS ? kFourPi : 1.f);
        const float x = k1 * k.z * p[e];
        const float y = __builtin_fmaf(k21 * x, x, x);
        const float amp = AXIS ? 1.f : lds.c[wv][n].x;
        am[e] = AXIS ? 1.f + y : __builtin_fmaf(amp, y, amp);
      } else {
        const float2 a = AXIS ? make_float2(1.f, k.z) : lds.c[wv][n];
        am[e] = __builtin_fmaf(a.y, p[e], a.x);
      }
    }
  }
};

// One step of 16 sources into the hi products' sums (Dr, Di) and the rest's (Lr, Li).
template <bool NEAR, int SIGN, bool OBL>
__device__ __forceinline__ void point_step(const PointWave<SIGN, OBL>& pw, int s, pf16& Dr,
                                           pf16& Di, pf16& Lr, pf16& Li) {
  constexpr float kSig = SIGN > 0 ? -1.f : 1.f;
  float yc[8], ys[8], q[8], ya[8], xc[8], xs[8], p[8], xa[8], g[8];
  pw.template phasors<NEAR, 1>(s, yc, ys, q, ya, g);
  pw.template phasors<NEAR, 0>(s, xc, xs, p, xa, g);
  Cplx8 y, x;
  float xr[8], xi[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    xr[e] = formed(xa[e] * xc[e]);
    xi[e] = formed(xa[e] * xs[e]);
  }
  split8(xr, pw.one, x.rh, x.rl);
  split8(xi, pw.one, x.ih, x.il);
  split8(yc, ya, y.rh, y.rl);
  split8(ys, ya, y.ih, y.il);
  cmul_lo(x, y, Lr, Li);
  cmul_hi(x, y, Dr, Di);
  if constexpr (!NEAR) {
    const ph8 ph = half8(p), qh = half8(q);
    Cplx8 a, b;  // p X and i sigma q Y
    a.rh = mul8(ph, x.rh);
    a.ih = mul8(ph, x.ih);
    b.rh = mul8(SIGN > 0 ? qh : neg8(qh), y.ih);
    b.ih = mul8(SIGN > 0 ? neg8(qh) : qh, y.rh);
    cmul_hi(a, b, Lr, Li);
  } else {
    constexpr float k11 = (OBL ? 1.f : 0.5f) / kFourPi;
    constexpr float kP = (float)SIGN * 9.424778f / kFourPi, kQ = kP / kFourPi;  // gP, gQ over id2 / w
    Cplx8 a, b;
    float yr[8], yi[8], br[8], bi[8];
    __builtin_amdgcn_sched_barrier(0);  // fewer live operands
#pragma unroll
    for (int e = 0; e < 8; ++e) {  // p X, g_1 Y
      yr[e] = ya[e] * yc[e];
      yi[e] = ya[e] * ys[e];
      const float gr = k11 * g[e] * g[e] * q[e], gi = q[e] * __builtin_fmaf(kQ * g[e], q[e], kSig);
      br[e] = formed(gr * yr[e] - gi * yi[e]);
      bi[e] = formed(gr * yi[e] + gi * yr[e]);
      xr[e] = formed(p[e] * xr[e]);
      xi[e] = formed(p[e] * xi[e]);
    }
    split8(br, pw.one, b.rh, b.rl);
    split8(bi, pw.one, b.ih, b.il);
    split8(xr, pw.one, a.rh, a.rl);
    split8(xi, pw.one, a.ih, a.il);
    cmul_lo(a, b, Lr, Li);
    cmul_hi(a, b, Lr, Li);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {  // p^2 X, g_2 Y
      const float q2 = q[e] * q[e];
      const float gr = -q2 * __builtin_fmaf(kSig * kQ * g[e], q[e], 0.5f), gi = kP * g[e] * q[e];
      br[e] = gr * yr[e] - gi * yi[e];
      bi[e] = gr * yi[e] + gi * yr[e];
      xr[e] *= p[e];
      xi[e] *= p[e];
    }
    b.rh = half8(br);
    b.ih = half8(bi);
    a.rh = half8(xr);
    a.ih = half8(xi);
    cmul_hi(a, b, Lr, Li);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {  // p^3 X, g_3 Y
      const float q2 = q[e] * q[e];
      const float gr = -kSig * kP * g[e] * q2, gi = (-kSig / 6.f) * (q2 * q[e]);
      br[e] = gr * yr[e] - gi * yi[e];
      bi[e] = gr * yi[e] + gi * yr[e];
      xr[e] *= p[e];
      xi[e] *= p[e];
    }
    b.rh = half8(br);
    b.ih = half8(bi);
    a.rh = half8(xr);
    a.ih = half8(xi);
    cmul_hi(a, b, Lr, Li);
  }
}

// The distance from the targets' plane to the nearest source's (0: inside).
__device__ __forceinline__ double plane_gap(double z, const PointPlan& pp) {
  return fmax(0.0, fmax(z - pp.hi[2], pp.lo[2] - z));
}

template <bool NEAR, int SIGN, bool OBL>
__device__ __forceinline__ void point_items(PointWave<SIGN, OBL>& pw, const PointPlan& pp,
                                            const PairTargets& pt, uint32_t S, uint32_t M,
                                            double inv_lambda, double2* __restrict__ out) {
  PointLds& lds = pw.lds;
  const uint32_t lane = pw.lane, wv = pw.wv, h = pw.h, j = pw.j;
  const uint32_t TI = (pt.nx + 31) / 32, TJ = (pt.ny + 31) / 32, items = TI * TJ * S;
  const uint32_t nb = (pp.n_slots + kPointBatch - 1) / kPointBatch, parts = kPairWaves * S;
  pw.kd = (double)j - (double)kPairMid;
  pw.kf = (float)j - kPairMid;
  pw.quad[0] = (float)(pw.kd * pw.kd * pt.px * pt.px);
  pw.quad[1] = (float)(pw.kd * pw.kd * pt.py * pt.py);
  pw.quad64[0] = pw.kd * pt.px * pt.px;
  pw.quad64[1] = pw.kd * pt.py * pt.py;
  const double gap = plane_gap(pt.z, pp), igap = 1.0 / gap;
  for (uint32_t item = blockIdx.x; item < items; item += gridDim.x) {
    const uint32_t split = item % S, tile = item / S;
    const uint32_t I = tile / TJ, J = tile - I * TJ;
    const double tcx = pt.x0 + ((double)(32 * I) + (double)kPairMid) * pt.px;
    const double tcy = pt.y0 + ((double)(32 * J) + (double)kPairMid) * pt.py;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      lds.re[wv][r][lane] = 0.0;
      lds.im[wv][r][lane] = 0.0;
    }
    for (uint32_t b = split * kPairWaves + wv; b < nb; b += parts) {
      // one source's constants per lane
      float unit;
      {
        const uint32_t slot = b * kPointBatch + lane;
        const int32_t n = slot < pp.n_slots ? pp.perm[slot] : -1;
        const size_t m = n < 0 ? 0 : (size_t)n;  // a padding slot: source 0, weight 0
        const float2 wt = n < 0 ? make_float2(0.f, 0.f) : pp.wc[slot];
        const double rx = tcx - pp.u[3 * m], ry = tcy - pp.u[3 * m + 1], rz = pt.z - pp.u[3 * m + 2];
        double d, id;
        hm_sqrt_inv(__builtin_fma(rz, rz, __builtin_fma(ry, ry, rx * rx)), d, id);
        const double al = 0.5 * id * inv_lambda;
        const double ax = 2.0 * rx * pt.px, ay = 2.0 * ry * pt.py;
        const float idf = (float)id, alf = (float)al;
        const float w = 0.5f * idf * __builtin_amdgcn_sqrtf(alf);
        const float A = (float)gap * (OBL ? (float)__builtin_fabs(rz) * idf * idf : idf);
        const float amp = A * wt.x;
        float mx = fabsf(amp);
        for (int off = 32; off; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        int e2 = 0;
        if (mx > 0.f && __builtin_isfinite(mx)) frexpf(mx, &e2);
        e2 = e2 < -126 ? -126 : (e2 > 127 ? 127 : e2);
        unit = ldexpf(1.f, e2);
        wave_sync();  // the previous batch's reads are done
        lds.a1[wv][lane] = make_double2(al * ax, al * ay);
        // odd batches enter the matrix cores with the opposite sign
        lds.f[wv][lane] =
            make_double2(al, kCycles32 + frac_cycle(d * inv_lambda) +
                                 ((double)(SIGN > 0 ? wt.y : -wt.y) + (b & 1 ? 0.5 : 0.0)));
        const float g = idf * idf * __builtin_amdgcn_rcpf(w), k1 = (OBL ? -1.f : -0.5f) * g;
        const float a0 = ldexpf(amp, -e2);
        lds.p1[wv][lane] = make_float4(w * (float)ax, kFourPi * w * (float)ay,
                                       NEAR ? g : (1.f / kFourPi) * k1, w);
        lds.c[wv][lane] = make_float2(a0, a0 * k1);
        wave_sync();
      }
      pf16 Dr = kZero16, Di = kZero16, Lr = kZero16, Li = kZero16;
#pragma unroll 1
      for (int s = 0; s < kPointBatch / 16; ++s) point_step<NEAR, SIGN, OBL>(pw, s, Dr, Di, Lr, Li);
      if (b & 1) unit = -unit;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        lds_add(&lds.re[wv][r][lane], (double)(unit * (Dr[r] + Lr[r])));
        lds_add(&lds.im[wv][r][lane], (double)(unit * (Di[r] + Li[r])));
      }
    }
    __syncthreads();
    // wave v adds up and writes registers 4 v .. 4 v + 3 of the waves' sums
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
      yr *= igap;
      yi *= igap;
      if (row < pt.nx && col < pt.ny) dst[(size_t)row * pt.ny + col] = make_double2(yr, yi);
      if (tile == 0 && r == 0) {  // copies of target 0 after the lattice
        const double cr = lane_f64(yr, 0), ci = lane_f64(yi, 0);
        for (uint32_t m = pt.nx * pt.ny + lane; m < M; m += 64) dst[m] = make_double2(cr, ci);
      }
    }
    __syncthreads();  // the sums are read before the next item clears them
  }
}

// Persistent, as k_superpose_pairs; handled: 1 when this kernel computes the call,
// 0 when the tiled (or 8 x 8) kernel has to.
template <int SIGN, bool OBL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, 2))) void
k_superpose_points(PointPlan pp, const PairTargets* __restrict__ ptp,
                   const uint32_t* __restrict__ flags, uint32_t n_flags, uint32_t* handled,
                   uint32_t S, uint32_t M, double inv_lambda, double2* __restrict__ out) {
  __shared__ PointLds lds;
  const PairTargets pt = *ptp;
  bool good = pt.mode != 0u;
  for (uint32_t k = threadIdx.x; k < n_flags; k += kBlock) good = good && flags[k] != 0u;
  const bool ok = __syncthreads_and(good ? 1 : 0) != 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *handled = ok ? 1u : 0u;
  if (!ok) return;  // uniform
  PointWave<SIGN, OBL> pw{lds, threadIdx.x & 63,
                          (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                          (threadIdx.x & 63) >> 5, threadIdx.x & 31};
  pw.one = 1.f;
  __asm__("" : "+v"(pw.one));
  if (pt.mode == kPairNear)
    point_items<true, SIGN, OBL>(pw, pp, pt, S, M, inv_lambda, out);
  else
    point_items<false, SIGN, OBL>(pw, pp, pt, S, M, inv_lambda, out);
}

// Whether this workgroup's share (b of n_probe) of the weights is finite in FP32.
__device__ bool weights_finite(const PointPlan& pp, int wf, const double* __restrict__ w0,
                               const double* __restrict__ w1, uint32_t b, uint32_t n_probe) {
  bool ok = true;
  for (uint32_t n = b * kBlock + threadIdx.x; n < pp.n; n += n_probe * kBlock) {
    const double x = wf == kPolar ? w0[n] : w0[2 * (size_t)n];
    const double y = wf == kPolar ? w1[n] : w0[2 * (size_t)n + 1];
    ok = ok && __builtin_isfinite((float)x) &&
         __builtin_isfinite(wf == kPolar ? y : (double)(float)y);
  }
  return ok;
}

// The polar weights of the slots (launch_tile_weights), and in the workgroups after
// those the targets' lattice.  A call with a weight that is not finite keeps the tiled
// kernel, whose infinities and NaN are those of the FP32 products: the integer phases
// here would turn a NaN into a number, and an f16 pair an infinity into NaN.
__global__ __launch_bounds__(kBlock) void k_point_prep(PointPlan pp, int wf,
                                                       const double* __restrict__ w0,
                                                       const double* __restrict__ w1,
                                                       const double* __restrict__ v, uint32_t M,
                                                       uint32_t n_probe, double inv_lambda,
                                                       uint32_t obl, PairTargets* pt,
                                                       uint32_t* flags) {
  __shared__ uint32_t s_min[kPairWaves];
  const uint32_t wb = (pp.n_slots + kBlock - 1) / kBlock;
  if (blockIdx.x < wb) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s < pp.n_slots) pp.wc[s] = slot_weight_polar(wf, w0, w1, pp.perm[s]);
    return;
  }
  const uint32_t b = blockIdx.x - wb;
  probe_targets(v, M, b, n_probe, pt, flags, s_min, weights_finite(pp, wf, w0, w1, b, n_probe),
                [&](const PairTargets& t, double cx0, double cx1, double cy0, double cy1) {
                  const auto far = [](double a0, double a1, double b0, double b1) {
                    return fmax(fabs(fmax(a0, a1) - b0), fabs(b1 - fmin(a0, a1)));
                  };
                  const double gap = plane_gap(t.z, pp);
                  const PairTerms d =
                      pair_terms((float)far(cx0, cx1, pp.lo[0], pp.hi[0]),
                                 (float)far(cy0, cy1, pp.lo[1], pp.hi[1]),
                                 (float)((double)kPairMid * fabs(t.px)),
                                 (float)((double)kPairMid * fabs(t.py)), 1.f / (float)gap,
                                 (float)inv_lambda);
                  return pair_far(d, obl != 0, 1.2e-3f) ? kPairFar
                         : pair_near(d, 0.07f)          ? kPairNear
                                                        : 0u;
                });
}

int point_splits(size_t M, size_t n_slots) {
  return pair_splits(M, (n_slots + 2 * kPointBatch - 1) / (2 * kPointBatch));
}

hipError_t launch_superpose_points(int sign, bool obliquity, const PointPlan& pp, WeightForm wf,
                                   const double* w0, const double* w1, const double* v, size_t M,
                                   double lambda, int S, PairTargets* pt, uint32_t* flags,
                                   uint32_t* handled, double2* out, hipStream_t stream) {
  if (M == 0 || !pp.n_slots) return hipErrorInvalidValue;
  // (eight sources a lane: one workgroup looked at 212040 weights for 66 us)
  const uint32_t n_probe = (uint32_t)std::min<size_t>(
      std::max<size_t>({M / kBlock, pp.n / (8 * kBlock), 1}), kPairFlags);
  const double il = 1.0 / lambda;
  k_point_prep<<<(pp.n_slots + kBlock - 1) / kBlock + n_probe, kBlock, 0, stream>>>(
      pp, (int)wf, w0, w1, v, (uint32_t)M, n_probe, il, obliquity ? 1u : 0u, pt, flags);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const size_t tiles = (M / 1024 + 1) * 4;
  const unsigned grid = (unsigned)std::min<size_t>(tiles * (size_t)S, kPairSlots);
  with_sign(sign, [&](auto sg) {
    with_bool(obliquity, [&](auto obl) {
      k_superpose_points<sg.value, (bool)obl.value><<<grid, kBlock, 0, stream>>>(
          pp, pt, flags, n_probe, handled, (uint32_t)S, (uint32_t)M, il, out);
    });
  });
  return hipGetLastError();
}

}  // namespace holo
