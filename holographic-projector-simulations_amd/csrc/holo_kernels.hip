// Hand-written gfx950 kernels for the Huygens point-source superposition
//   y_m = sum_n a_n / d_nm * exp(i (phi_n +/- 2 pi d_nm / lambda))
// (cuda/superposition.cu:35-154 computes the same sum with per_block and a
// CUB/cuBLAS reduction; these kernels are a new design for CDNA4):
//
// * One lane owns R targets; their positions and FP64 accumulators stay in
//   VGPRs for the whole launch.
// * The source index is wave-uniform, so source data is fetched with scalar
//   loads into SGPRs and broadcast to all 64 lanes for free -- no LDS and no
//   per-lane source traffic.
// * Sources are split into S contiguous chunks (blockIdx.y) only when the
//   target count alone cannot fill the 256 CUs; the S partial fields are
//   summed afterwards in a fixed order, so results are deterministic.
// * No MFMA: the sum is not a contraction; it is bound by VALU and
//   transcendental issue.
#include <hip/hip_runtime.h>
#include <math.h>

#include "holo_device.hpp"
#include "holo_internal.hpp"
#include "holo_mc.hpp"

namespace holo {

Tuning& tuning() {
  static Tuning t;
  return t;
}

// f64_shape's estimates, in ns, from sweeps of R and S over 1e6 .. 4e10 pairs
// (lattice sources; within 5 % of the measured times from 2e8 pairs up).  A SIMD
// that takes c waves one after the other or together needs w (c + k), w = a wave's
// pairs at kF64Pair[R] each and k the last wave's latency that nothing hides; c is
// the largest count of workgroups per CU.  A workgroup loads the sin/cos table
// (kF64Start for every kF64Resident of them on a CU: fitted, like the rest; 4 or 5
// workgroups are resident, by the layout's variant), and a split writes partial values
// that a reduction reads.
struct F64Cost {
  int R;
  double pair, k;
};
constexpr F64Cost kF64Cost[] = {{4, 58.5, 0.475}, {2, 59.4, 0.75}, {1, 62.6, 1.62}};
constexpr double kF64Start = 1500, kF64Reduce = 3000, kF64Partial = 0.008;
constexpr size_t kF64Cus = 256, kF64Resident = 5;
constexpr size_t kF64MinSources = 32;  // per split

int choose_splits(size_t M, int R, size_t units, size_t min_units, size_t max_splits) {
  const Tuning& tu = tuning();
  if (tu.splits > 0) return (int)std::min<size_t>(tu.splits, std::max<size_t>(units, 1));
  const size_t waves = (M + 64 * R - 1) / (64 * R);
  size_t S = (tu.target_waves + waves - 1) / std::max<size_t>(waves, 1);
  const size_t max_by_units = std::max<size_t>(units / std::max<size_t>(min_units, 1), 1);
  S = std::min(S, max_by_units);
  S = std::min<size_t>(S, max_splits);
  return (int)std::max<size_t>(S, 1);
}

int tile_splits(size_t M, int R, size_t n_tiles) {
  if (!n_tiles) return 1;
  return choose_splits(M, R, n_tiles, M < kFillTargets * R ? 1 : 64, kTileSplits);
}

// 1024 sources on 4096 targets: 367 us as 4 workgroups, 15 us by this rule; 7680 on
// 30000: 499 and 270 us; 65536 on 262144: 15.7 ms (16 splits) and 15.1 - 15.7 ms.
// Launch shape of the FP64 kernel: the targets per lane R (at most r_f64) and source
// splits S of the smallest estimated time, S M at most `cap` partial values (unless
// S = 1).  With `splits` set by the caller R = r_f64 and S = splits.
F64Shape f64_shape(size_t M, size_t N, size_t cap) {
  const Tuning& tu = tuning();
  const int top = tu.r_f64 == 1 || tu.r_f64 == 4 ? tu.r_f64 : 2;
  F64Shape best{top, 1};
  if (N == 0 || M == 0) return best;
  if (tu.splits > 0) {
    best.S = (int)std::min<size_t>((size_t)tu.splits, N);
    while (best.S > 1 && (size_t)best.S * M > cap) --best.S;
    return best;
  }
  double least = 1e300;
  for (const F64Cost& f : kF64Cost) {
    if (f.R > top) continue;
    const size_t tb = (M + (size_t)kBlock * f.R - 1) / ((size_t)kBlock * f.R);
    for (const int S : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 40, 48, 64, 96, 128}) {
      const size_t blocks = tb * (size_t)S, c = (blocks + kF64Cus - 1) / kF64Cus;
      if (S > 1 && ((size_t)S * M > cap || N < (size_t)S * kF64MinSources ||
                    blocks > (size_t)tu.target_waves))
        break;
      const double w = (double)((N + S - 1) / S) * f.R * f.pair;
      double t = w * ((double)c + f.k) + kF64Start * (double)((c + kF64Resident - 1) / kF64Resident);
      if (S > 1) t += kF64Reduce + (double)S * (double)M * kF64Partial;
      if (t < least) {
        least = t;
        best = F64Shape{f.R, S};
      }
    }
  }
  return best;
}

// ---------------------------------------------------------------------------
// FP64 brute force.

// PZ: every source has the z of source 0, so dz = vz - uz is formed once per
// target (the same bits as per pair).
// ROWS (with PZ): from source `first` on, the sources come in rows of `row`
// consecutive sources that share one x, and those before it (of this split) share
// one too (a lattice in x-slow order, cuda/init.h:89-158), so dx^2 is formed once
// per (target, row): again the same bits as per pair.
// s_tab: the sin/cos table, already in LDS.
template <int SIGN, int R, int WF, int MATH, bool OBL, bool PZ, bool ROWS>
__device__ __forceinline__ void superpose_f64_body(
    const double* __restrict__ w0, const double* __restrict__ w1,
    const double* __restrict__ u, uint32_t N, uint32_t chunk, uint32_t first, uint32_t row,
    const double* __restrict__ v, uint32_t M, double K,
    double2* __restrict__ out, const double* s_tab) {
  static_assert(!ROWS || PZ, "rows need sources in one plane");
  const uint32_t n0 = blockIdx.y * chunk;
  const uint32_t n1 = min(N, n0 + chunk);
  const uint32_t base = blockIdx.x * (kBlock * R) + threadIdx.x;
  double vx[R], vy[R], vz[R], ar[R], ai[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t m = base + r * kBlock;
    const size_t mm = m < M ? m : M - 1;
    vx[r] = v[3 * mm];
    vy[r] = v[3 * mm + 1];
    vz[r] = v[3 * mm + 2];
    ar[r] = 0.0;
    ai[r] = 0.0;
  }
  double dz0[R];
#pragma unroll
  for (int r = 0; r < R; ++r) dz0[r] = PZ && n0 < n1 ? vz[r] - u[3 * (size_t)n0 + 2] : 0.0;
  // sources [a, b); with ROWS their dx^2 per target is dxx
  auto sources = [&](uint32_t a, uint32_t b, const double(&dxx)[R]) {
    for (uint32_t n = a; n < b; ++n) {
      const double ux = ROWS ? 0.0 : u[3 * (size_t)n];
      const double uy = u[3 * (size_t)n + 1];
      const double uz = PZ ? 0.0 : u[3 * (size_t)n + 2];
      if constexpr (WF == kPolar) {
        const double a = w0[n];
        const double phi = w1[n];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const double dy = vy[r] - uy, dz = PZ ? dz0[r] : vz[r] - uz;
          PairF64 p;
          if constexpr (ROWS)
            p = pair_f64_s<SIGN, MATH, OBL>(a, phi, dxx[r], dy, dz, K);
          else
            p = pair_f64_d<SIGN, MATH, OBL>(a, phi, vx[r] - ux, dy, dz, K);
          accumulate_phasor<MATH>(p.r, p.arg, ar[r], ai[r], s_tab);
        }
      } else {
        const double wr = w0[2 * (size_t)n];
        const double wi = w0[2 * (size_t)n + 1];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const double dx = vx[r] - ux, dy = vy[r] - uy, dz = PZ ? dz0[r] : vz[r] - uz;
          double d, id;
          hm_sqrt_inv(__builtin_fma(dz, dz, __builtin_fma(dy, dy, ROWS ? dxx[r] : dx * dx)),
                      d, id);
          if constexpr (OBL) id *= __builtin_fabs(dz) * id;
          const double arg = (SIGN > 0 ? d : -d) * K;
          double s, c;
          if constexpr (MATH == 0) {
            hm_sincos(arg, s_tab, s, c);
          } else {
            sincos(arg, &s, &c);
          }
          c *= id;
          s *= id;
          ar[r] += wr * c - wi * s;
          ai[r] += wr * s + wi * c;
        }
      }
    }
  };
  if constexpr (ROWS) {
    for (uint32_t n = n0; n < n1;) {
      // end of n's row
      const uint32_t e = min(n1, n < first ? first : first + ((n - first) / row + 1) * row);
      const double ux = u[3 * (size_t)n];
      double dxx[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double dx = vx[r] - ux;
        dxx[r] = dx * dx;
      }
      sources(n, e, dxx);
      n = e;
    }
  } else {
    const double none[R] = {};
    sources(n0, n1, none);
  }
  double2* dst = out + (size_t)blockIdx.y * M;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t m = base + r * kBlock;
    if (m < M) dst[m] = make_double2(ar[r], ai[r]);
  }
}

// The sin/cos table, 32 KB, into LDS (5 workgroups per CU, as the VGPRs allow).
constexpr int kTab = sizeof(kSinCosTab) / sizeof(double);
static_assert(kTab % kBlock == 0, "table copy");

__device__ __forceinline__ void load_sincos_table(double* s_tab) {
#pragma unroll
  for (int q = 0; q < kTab / kBlock; ++q)
    s_tab[threadIdx.x + q * kBlock] = kSinCosTab[threadIdx.x + q * kBlock];
  __syncthreads();
}

template <int SIGN, int R, int WF, int MATH, bool OBL, bool PZ, bool ROWS>
__global__ __launch_bounds__(kBlock) void k_superpose_f64(
    const double* __restrict__ w0, const double* __restrict__ w1,
    const double* __restrict__ u, uint32_t N, uint32_t chunk, uint32_t row,
    const double* __restrict__ v, uint32_t M, double K,
    double2* __restrict__ out) {
  __shared__ double s_tab[kTab];
  load_sincos_table(s_tab);
  superpose_f64_body<SIGN, R, WF, MATH, OBL, PZ, ROWS>(w0, w1, u, N, chunk, 0u, row, v, M, K,
                                                        out, s_tab);
}

// The same sum for sources whose layout the host has not scanned (device
// pointers; the host-pointer and plan paths scan the positions on the host): every
// workgroup looks at the sources of its own split first, which takes a few loads a
// lane against 60 ns per source and target of a wave, and no launch.
// allow: bit 0 = look for one z, bit 1 = look for rows too.  Returns 3 (one z, and
// rows of at least 4 from `first`, the last one possibly shorter), 1 (one z) or 0.
// s_w: 4 words of LDS.
__device__ uint32_t split_layout(const double* __restrict__ u, uint32_t n0, uint32_t n1,
                                 uint32_t allow, uint32_t* s_w, uint32_t& first,
                                 uint32_t& row) {
  first = row = n1;
  if (!(allow & 1u) || n0 >= n1) return 0u;
  if (threadIdx.x < 4) s_w[threadIdx.x] = threadIdx.x < 2 ? n1 : 0u;
  __syncthreads();
  const double x0 = u[3 * (size_t)n0], z0 = u[3 * (size_t)n0 + 2];
  bool planar = true;
  uint32_t hit = n1;  // the first source with another x
  for (uint32_t n = n0 + threadIdx.x; n < n1; n += kBlock) {
    planar = planar && u[3 * (size_t)n + 2] == z0;
    if (hit == n1 && u[3 * (size_t)n] != x0) hit = n;
  }
  if (hit < n1) atomicMin(&s_w[0], hit);
  if (!planar) s_w[2] = 1u;
  __syncthreads();
  if (s_w[2]) return 0u;
  if (!(allow & 2u)) return 1u;
  first = __builtin_amdgcn_readfirstlane(s_w[0]);  // (scalar: the loops' bounds)
  if (first == n1) return 3u;  // one x
  const double x1 = u[3 * (size_t)first];
  for (uint32_t n = first + threadIdx.x; n < n1; n += kBlock)
    if (u[3 * (size_t)n] != x1) {
      atomicMin(&s_w[1], n);
      break;
    }
  __syncthreads();
  row = __builtin_amdgcn_readfirstlane(s_w[1]) - first;
  bool rows = row >= 4;
  if (rows)
    for (uint32_t n = first + threadIdx.x; n < n1; n += kBlock)
      rows = rows && u[3 * (size_t)n] == u[3 * (size_t)(n - (n - first) % row)];
  if (!rows) s_w[3] = 1u;
  __syncthreads();
  return s_w[3] ? 1u : 3u;
}

// The branch is uniform over the workgroup, and every branch gives the same bits.
// 98 VGPRs, 4 waves a SIMD: held to 96 for 5 it was up to 3 % slower.
template <int SIGN, int R, int WF, bool OBL>
__global__ __launch_bounds__(kBlock) void k_superpose_f64_auto(
    const double* __restrict__ w0, const double* __restrict__ w1,
    const double* __restrict__ u, uint32_t N, uint32_t chunk, uint32_t allow,
    const double* __restrict__ v, uint32_t M, double K, double2* __restrict__ out) {
  __shared__ double s_tab[kTab];  // 32 KB: with any more LDS only 4 workgroups fit a CU
  uint32_t first, row;
  const uint32_t n0 = min(N, blockIdx.y * chunk);
  const uint32_t mode = split_layout(u, n0, min(N, n0 + chunk), allow,
                                     reinterpret_cast<uint32_t*>(s_tab), first, row);
  __syncthreads();
  load_sincos_table(s_tab);
  if (mode == 3u)
    superpose_f64_body<SIGN, R, WF, 0, OBL, true, true>(w0, w1, u, N, chunk, first, row, v, M, K,
                                                        out, s_tab);
  else if (mode == 1u)
    superpose_f64_body<SIGN, R, WF, 0, OBL, true, false>(w0, w1, u, N, chunk, 0u, 0u, v, M, K,
                                                         out, s_tab);
  else
    superpose_f64_body<SIGN, R, WF, 0, OBL, false, false>(w0, w1, u, N, chunk, 0u, 0u, v, M, K,
                                                          out, s_tab);
}

// The splits to sum (`handled`: launch_reduce_partials).
__device__ __forceinline__ uint32_t splits_of(const uint32_t* handled, uint32_t Sp, uint32_t S) {
  return handled && *handled ? Sp : S;
}

// One thread per target, the splits in order, eight loads in flight.
__global__ __launch_bounds__(kBlock) void k_reduce_partials(
    const double2* __restrict__ partial, const uint32_t* __restrict__ handled, uint32_t Sp,
    uint32_t Sg, uint32_t M, double2* __restrict__ y) {
  const uint32_t S = splits_of(handled, Sp, Sg);
  if (S <= 1) return;  // that split wrote y
  const uint32_t m = blockIdx.x * kBlock + threadIdx.x;
  if (m < M) y[m] = sum_splits(partial + m, S, M);
}

// Fewer targets than fill the GPU: 32 targets by 8 ranges of splits per workgroup,
// each range summed in order, then the ranges.
__global__ __launch_bounds__(kBlock) void k_reduce_partials_few(
    const double2* __restrict__ partial, const uint32_t* __restrict__ handled, uint32_t Sp,
    uint32_t Sg, uint32_t M, double2* __restrict__ y) {
  __shared__ double2 s_part[8][32];
  const uint32_t S = splits_of(handled, Sp, Sg);
  if (S <= 1) return;
  const uint32_t t = threadIdx.x & 31, q = threadIdx.x >> 5;
  const uint32_t m = blockIdx.x * 32 + t;
  const uint32_t a = q * S / 8, b = (q + 1) * S / 8;
  if (m < M) s_part[q][t] = sum_splits(partial + (size_t)a * M + m, b - a, M);
  __syncthreads();
  if (q == 0 && m < M) {
    double2 r = s_part[0][t];
    for (int k = 1; k < 8; ++k) {
      r.x += s_part[k][t].x;
      r.y += s_part[k][t].y;
    }
    y[m] = r;
  }
}

// Few targets over many splits (the error report's 256 targets over up to
// 1024 splits): one workgroup per target, lane t summing the splits t, t + 256,
// ... in order, then a fixed tree over the lanes, so the order is set by S
// alone.
__global__ __launch_bounds__(kBlock) void k_reduce_partials_wide(
    const double2* __restrict__ partial, const uint32_t* __restrict__ handled, uint32_t Sp,
    uint32_t Sg, uint32_t M, double2* __restrict__ y) {
  __shared__ double s_re[kBlock], s_im[kBlock];
  const uint32_t S = splits_of(handled, Sp, Sg);
  if (S <= 1) return;
  const uint32_t m = blockIdx.x, t = threadIdx.x;
  double re = 0.0, im = 0.0;
  for (uint32_t s = t; s < S; s += kBlock) {
    const double2 p = partial[(size_t)s * M + m];
    re += p.x;
    im += p.y;
  }
  s_re[t] = re;
  s_im[t] = im;
  __syncthreads();
  for (uint32_t h = kBlock / 2; h > 0; h >>= 1) {
    if (t < h) {
      s_re[t] += s_re[t + h];
      s_im[t] += s_im[t + h];
    }
    __syncthreads();
  }
  if (t == 0) y[m] = make_double2(s_re[0], s_im[0]);
}

// Up to this many targets one thread each leaves most of the GPU idle (30000
// targets, 64 splits: 17.9 us; by ranges 5.5 us).
constexpr size_t kReduceFew = 131072;

// The form is chosen by S, so that a call's bits do not depend on a path that was
// tried before (Sp splits, when *handled).
hipError_t launch_reduce_partials(int S, size_t M, const double2* partial, double2* y,
                                  hipStream_t stream, const uint32_t* handled, int Sp) {
  if (!handled) Sp = S;
  if (std::max(S, Sp) <= 1 || M == 0) return hipSuccess;
  const size_t by = S > 1 ? S : Sp;
  const uint32_t s = (uint32_t)S, sp = (uint32_t)Sp, m = (uint32_t)M;
  if (M <= 4096 && by >= 64)
    k_reduce_partials_wide<<<m, kBlock, 0, stream>>>(partial, handled, sp, s, m, y);
  else if (M <= kReduceFew && by >= 8)
    k_reduce_partials_few<<<(m + 31) / 32, kBlock, 0, stream>>>(partial, handled, sp, s, m, y);
  else
    k_reduce_partials<<<(unsigned)((M + kBlock - 1) / kBlock), kBlock, 0, stream>>>(
        partial, handled, sp, s, m, y);
  return hipGetLastError();
}

hipError_t launch_superpose_f64(int sign, WeightForm wf, bool obliquity, bool uniform_z,
                                size_t row, const double* w0, const double* w1, const double* u,
                                size_t N,
                                const double* v, size_t M, double K,
                                double2* y, double2* partial,
                                size_t partial_cap, hipStream_t stream, bool few_targets) {
  if (M == 0) return hipSuccess;
  F64Shape shape = f64_shape(M, N, partial_cap);
  if (few_targets) {
    shape = F64Shape{1, N ? choose_splits(M, 1, N, 128, kFewTargetSplits) : 1};
    while (shape.S > 1 && (size_t)shape.S * M > partial_cap) --shape.S;
  }
  const int R = shape.R, S = shape.S;
  const uint32_t chunk = N ? (uint32_t)((N + S - 1) / S) : 0;
  const dim3 grid((unsigned)((M + (size_t)kBlock * R - 1) / ((size_t)kBlock * R)),
                  (unsigned)S);
  double2* out = S > 1 ? partial : y;
  with_sign(sign, [&](auto sg) {
    with_r(R, [&](auto rr) {
      with_bool(wf == kCartesian, [&](auto cart) {
        with_bool(obliquity, [&](auto obl) {
          constexpr int wfv = cart.value ? kCartesian : kPolar;
          if (tuning().f64_libm) {
            k_superpose_f64<sg.value, rr.value, wfv, 1, (bool)obl.value, false, false>
                <<<grid, kBlock, 0, stream>>>(w0, w1, u, (uint32_t)N, chunk, 0u, v,
                                              (uint32_t)M, K, out);
          } else if (uniform_z && tuning().f64_planar && row && tuning().f64_rows) {
            k_superpose_f64<sg.value, rr.value, wfv, 0, (bool)obl.value, true, true>
                <<<grid, kBlock, 0, stream>>>(w0, w1, u, (uint32_t)N, chunk, (uint32_t)row, v,
                                              (uint32_t)M, K, out);
          } else {
            with_bool(uniform_z && tuning().f64_planar, [&](auto pz) {
              k_superpose_f64<sg.value, rr.value, wfv, 0, (bool)obl.value, (bool)pz.value, false>
                  <<<grid, kBlock, 0, stream>>>(w0, w1, u, (uint32_t)N, chunk, 0u, v,
                                                (uint32_t)M, K, out);
            });
          }
        });
      });
    });
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_reduce_partials(S, M, partial, y, stream);
}

hipError_t launch_superpose_f64_auto(int sign, WeightForm wf, bool obliquity,
                                     const double* w0, const double* w1, const double* u,
                                     size_t N, const double* v, size_t M, double K, double2* y,
                                     double2* partial, size_t partial_cap,
                                     hipStream_t stream) {
  if (M == 0) return hipSuccess;
  // the options switch the paths off as they do for host-scanned sources
  const uint32_t allow = tuning().f64_planar ? (tuning().f64_rows ? 3u : 1u) : 0u;
  const F64Shape shape = f64_shape(M, N, partial_cap);
  const int R = shape.R, S = shape.S;
  const uint32_t chunk = N ? (uint32_t)((N + S - 1) / S) : 0;
  const dim3 grid((unsigned)((M + (size_t)kBlock * R - 1) / ((size_t)kBlock * R)),
                  (unsigned)S);
  double2* out = S > 1 ? partial : y;
  with_sign(sign, [&](auto sg) {
    with_r(R, [&](auto rr) {
      with_bool(wf == kCartesian, [&](auto cart) {
        with_bool(obliquity, [&](auto obl) {
          constexpr int wfv = cart.value ? kCartesian : kPolar;
          k_superpose_f64_auto<sg.value, rr.value, wfv, (bool)obl.value>
              <<<grid, kBlock, 0, stream>>>(w0, w1, u, (uint32_t)N, chunk, allow, v,
                                            (uint32_t)M, K, out);
        });
      });
    });
  });
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_reduce_partials(S, M, partial, y, stream);
}

// ---------------------------------------------------------------------------
// FP32-split brute force over tiles of T sources.
//
// Per (target, tile), in FP64: r = v - c, d_ref = |r|, the fractional cycle
// f = frac(d_ref / lambda), and the tile rotation e^{i sign 2 pi f}.
// Per pair, in FP32 and without cancellation:
//   q = |delta|^2 - 2 r.delta          (= d^2 - d_ref^2, delta = u - c)
//   t = (d - d_ref) / lambda = q (alpha + c2 q)        to O(q^3), with
//       alpha = 1 / (2 d_ref lambda),  c2 = -1 / (8 d_ref^3 lambda)
//   1/d = 1/d_ref + q g,  g = -1 / (2 d_ref^3)          to O(q^2)
//   term = w * e^{i sign 2 pi t} / d
// (d = sqrt(d_ref^2 + q) = d_ref + q/(2 d_ref) - q^2/(8 d_ref^3) + ...).  The
// T terms of a tile are summed in FP32, rotated by the tile's FP64-derived
// phase and added into FP64 accumulators.  PLANAR: every slot of every tile
// has delta_z = 0 (sources on planes z = const), so the z term of q drops.
// Valid in the far field of each tile: |q| / d_ref^2 << 1 (tile radius much
// smaller than the distance) and |t| of order one cycle.

template <int SIGN, int R, int T, bool PLANAR, bool OBL>
__global__ __launch_bounds__(kBlock) void k_superpose_f32s(
    const double4* __restrict__ centre, const float4* __restrict__ geo,
    const float2* __restrict__ wc, const int32_t* __restrict__ perm,
    const double* __restrict__ u, uint32_t n_tiles, uint32_t chunk_tiles,
    const double* __restrict__ v, uint32_t M, double lambda,
    double inv_lambda, const uint32_t* __restrict__ skip, double2* __restrict__ out) {
  if (skip && *skip) return;
  const uint32_t t0 = blockIdx.y * chunk_tiles;
  const uint32_t t1 = min(n_tiles, t0 + chunk_tiles);
  const uint32_t base = blockIdx.x * (kBlock * R) + threadIdx.x;
  double vx[R], vy[R], vz[R], ar[R], ai[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t m = base + r * kBlock;
    const size_t mm = m < M ? m : M - 1;
    vx[r] = v[3 * mm];
    vy[r] = v[3 * mm + 1];
    vz[r] = v[3 * mm + 2];
    ar[r] = 0.0;
    ai[r] = 0.0;
  }
  for (uint32_t t = t0; t < t1; ++t) {
    const double4 c = centre[t];
    const float2 rho = __builtin_bit_cast(float2, c.w);  // lateral, axial tile radius
    float m2rx[R], m2ry[R], m2rz[R], alpha[R], c2[R], gq[R], invd[R], rzf[R];
    float ct[R], st[R], sr[R], si[R];
    bool near[R];
    bool any_near = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double rx = vx[r] - c.x, ry = vy[r] - c.y, rz = vz[r] - c.z;
      double dref, id;
      hm_sqrt_inv(__builtin_fma(rz, rz, __builtin_fma(ry, ry, rx * rx)), dref, id);
      {
        const float rxy = __builtin_sqrtf((float)__builtin_fma(ry, ry, rx * rx));
        const float qmax = 2.f * (rxy * rho.x + __builtin_fabsf((float)rz) * rho.y) +
                           rho.x * rho.x + rho.y * rho.y;
        const float ia = (float)(id * inv_lambda);  // 1 / (d lambda)
        const float idf = (float)id;
        const float round_err = 3e-8f * qmax * ia;
        const float trunc_err = 0.0625f * qmax * qmax * qmax * ia * idf * idf * idf * idf;
        // NaN (a target at the tile centre) also counts as near
        near[r] = !(round_err <= kGuardCycles && trunc_err <= 0.05f * kGuardCycles);
        any_near |= near[r];
      }
      const float f = (float)frac_cycle(dref * inv_lambda);
      sincos_rev_f32(f, st[r], ct[r]);
      m2rx[r] = (float)(-2.0 * rx);
      m2ry[r] = (float)(-2.0 * ry);
      m2rz[r] = (float)(-2.0 * rz);
      const double id2 = id * id;
      const double a = 0.5 * id * inv_lambda;
      alpha[r] = (float)a;
      c2[r] = (float)(-0.25 * a * id2);
      if constexpr (OBL) {
        // |dz| / d^2 = |dz| (1/d_ref^2 - q/d_ref^4 + O(q^2)); planar tiles
        // have dz = rz for every slot, so |rz| folds into the coefficients.
        const double zs = PLANAR ? __builtin_fabs(rz) : 1.0;
        invd[r] = (float)(zs * id2);
        gq[r] = (float)(-zs * id2 * id2);
        rzf[r] = (float)rz;
      } else {
        gq[r] = (float)(-0.5 * id2 * id);
        invd[r] = (float)id;
        rzf[r] = 0.f;
      }
      sr[r] = 0.f;
      si[r] = 0.f;
    }
    const float4* g = geo + (size_t)t * T;
    const float2* w = wc + (size_t)t * T;
    // a wave whose every target is near this tile skips the expansion
    bool all_near = true;
#pragma unroll
    for (int r = 0; r < R; ++r) all_near &= near[r];
    if (__builtin_amdgcn_ballot_w64(!all_near) != 0) {
#pragma unroll 4
      for (int j = 0; j < T; ++j) {
        const float4 gj = g[j];
        const float2 wj = w[j];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float q = __builtin_fmaf(m2ry[r], gj.y, gj.w);
          if constexpr (!PLANAR) q = __builtin_fmaf(m2rz[r], gj.z, q);
          q = __builtin_fmaf(m2rx[r], gj.x, q);
          // w e^{i s 2 pi t} = |w| e^{2 pi i (arg w + s t)}: the weight's phase
          // joins the pair's, its modulus the amplitude
          const float pc = __builtin_fmaf(c2[r], q, alpha[r]);
          const float tt = SIGN > 0 ? __builtin_fmaf(q, pc, wj.y) : __builtin_fmaf(-q, pc, wj.y);
          float sn, cs;
          sincos_rev_f32(tt, sn, cs);
          float amp = wj.x * __builtin_fmaf(q, gq[r], invd[r]);
          if constexpr (OBL && !PLANAR) amp *= __builtin_fabsf(rzf[r] - gj.z);
          sr[r] = __builtin_fmaf(amp, cs, sr[r]);
          si[r] = __builtin_fmaf(amp, sn, si[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double xr = near[r] ? 0.0 : sr[r], xi = near[r] ? 0.0 : si[r];
      const double cr = ct[r], cs = SIGN > 0 ? (double)st[r] : -(double)st[r];
      ar[r] += xr * cr - xi * cs;
      ai[r] += xr * cs + xi * cr;
    }
    if (any_near)  // thick tiles or near field
      exact_tile_pairs_polar<SIGN, OBL, R, PLANAR>(u, perm + (size_t)t * T, w, T, c.z, vx, vy,
                                                   vz, near, inv_lambda, ar, ai);
  }
  double2* dst = out + (size_t)blockIdx.y * M;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t m = base + r * kBlock;
    if (m < M) dst[m] = make_double2(ar[r], ai[r]);
  }
}

template <typename F>
static bool with_tile(unsigned T, F&& f) {
  switch (T) {
    case 8: f(IC<8>{}); return true;
    case 16: f(IC<16>{}); return true;
    case 32: f(IC<32>{}); return true;
    case 64: f(IC<64>{}); return true;
    default: return false;
  }
}

hipError_t launch_superpose_f32s(int sign, bool obliquity, const TileSet& ts,
                                 const float2* wc, const double* v, size_t M,
                                 double lambda, double2* y, double2* partial,
                                 size_t partial_cap, hipStream_t stream,
                                 const uint32_t* skip, int Sp) {
  if (M == 0) return hipSuccess;
  int R = tuning().r_f32;
  if (R != 1 && R != 2 && R != 4) R = 2;
  int S = tile_splits(M, R, ts.n_tiles);
  while (S > 1 && (size_t)S * M > partial_cap) --S;
  const uint32_t chunk = ts.n_tiles ? (ts.n_tiles + S - 1) / S : 0;
  const dim3 grid((unsigned)((M + (size_t)kBlock * R - 1) / ((size_t)kBlock * R)),
                  (unsigned)S);
  double2* out = S > 1 ? partial : y;
  const double il = 1.0 / lambda;
  const bool ok = with_tile(ts.tile, [&](auto tt) {
    with_sign(sign, [&](auto sg) {
      with_r(R, [&](auto rr) {
        with_bool(ts.planar, [&](auto pl) {
          with_bool(obliquity, [&](auto obl) {
            k_superpose_f32s<sg.value, rr.value, tt.value, (bool)pl.value, (bool)obl.value>
                <<<grid, kBlock, 0, stream>>>(ts.centre, ts.geo, wc, ts.perm, ts.u, ts.n_tiles,
                                              chunk, v, (uint32_t)M, lambda, il, skip, out);
          });
        });
      });
    });
  });
  if (!ok) return hipErrorInvalidValue;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_reduce_partials(S, M, partial, y, stream, skip, Sp);
}

__global__ __launch_bounds__(kBlock) void k_tile_weights(
    int wf, const double* __restrict__ w0, const double* __restrict__ w1,
    const int32_t* __restrict__ perm, uint32_t n_slots,
    float2* __restrict__ wc, int polar_out) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n_slots) return;
  wc[s] = polar_out ? slot_weight_polar(wf, w0, w1, perm[s]) : slot_weight(wf, w0, w1, perm[s]);
}

hipError_t launch_tile_weights(WeightForm wf, const double* w0,
                               const double* w1, const int32_t* perm,
                               size_t n_slots, float2* wc,
                               hipStream_t stream, bool polar_out) {
  if (!n_slots) return hipSuccess;
  const unsigned blocks = (unsigned)((n_slots + kBlock - 1) / kBlock);
  k_tile_weights<<<blocks, kBlock, 0, stream>>>((int)wf, w0, w1, perm,
                                               (uint32_t)n_slots, wc, polar_out ? 1 : 0);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Monte Carlo: target m draws K indices n_{m,k} from Philox4x32-10 keyed by
// the seed with counter (k/2, m, 0, kMcStream); words (x,y) serve even k,
// (z,w) odd k; Lemire multiply-shift maps 64 bits into [0, N).
// Batched ("shared") Monte Carlo: the targets of group g = m / kMcGroup share
// one subset, drawn with counter (k/2, g, kMcSharedTag, kMcStream); the
// index is then wave-uniform, Philox runs on the scalar unit and sources
// arrive through scalar loads.

constexpr uint32_t kMcSharedTag = 0x80000000u;

// The Philox block of draws k, k + 1 (k even) of target m: per target, or
// (SHARED_IDX) of m's group's shared subset.
template <bool SHARED_IDX>
__device__ __forceinline__ U4 mc_draws(uint32_t k, uint32_t m, uint32_t slo, uint32_t shi) {
  if constexpr (SHARED_IDX)
    return philox4x32_10(U4{k >> 1, m / kMcGroup, kMcSharedTag, kMcStream}, slo, shi);
  else
    return philox4x32_10<true>(U4{k >> 1, m, 0u, kMcStream}, slo, shi);
}

// A drawn source n as (x, y, z, w): w = amp (FP64, the phase in ph[n]) or the
// bit-cast FP32 weight (FP32-split).  On a product grid (FP32-split only) the
// sources of the leading complete rows come from the row and column tables
// and the weight array, the same values as the packed records: of a call's
// sources all (kMcTables), none (kMcRecords) or some (kMcMixed, which chooses
// each component's address by a select).
enum McView { kMcRecords, kMcStaged, kMcTables, kMcMixed };
constexpr uint32_t kMcTable = 2560;  // entries of the tables staged in LDS

struct McSourceView {
  const double4* pos;
  McLattice lat;
  uint32_t ny = 0, body = 0, magic = 0, row0 = 0;
  bool whole = false;  // all sources are on the grid
  double z = 0.0;
  const double* table = nullptr;
  __device__ McSourceView(const double4* p, const McLattice& l, bool fp64, uint32_t N)
      : pos(p), lat(l) {
    uint32_t rows = 0;
    if (!fp64 && lat.info) {
      ny = lat.info[0];
      rows = ny ? lat.info[1] : 0u;
      if (!rows) ny = 0;
    }
    body = min(rows * ny, N);
    whole = ny && body == N;
    if (!lat.use || body < N / 2) body = 0;  // jittered sources start with a "row" of one
    if (ny) {
      magic = 0xffffffffu / ny;
      z = lat.xy[kLatticeMaxRow];
    }
  }
  // Whether all sources are on the grid and the tables' part for any `width` of them
  // fits into kMcTable entries.
  __device__ __forceinline__ bool stages(uint32_t width) const {
    return whole && ny <= kMcTable && ny + width / ny + 2 <= kMcTable;
  }
  // The tables' part for the sources [lo, hi) into tab, the columns first; the whole
  // workgroup.
  __device__ __forceinline__ void stage(uint32_t lo, uint32_t hi, double* tab) {
    row0 = lo / ny;
    const uint32_t entries = ny + (hi - 1) / ny + 1 - row0;
    for (uint32_t k = threadIdx.x; k < entries; k += kBlock)
      tab[k] = k < ny ? lat.xy[k] : lat.xy[kLatticeMaxRow + 1 + row0 + k - ny];
    table = tab;
    __syncthreads();
  }
  template <McView VIEW>
  __device__ __forceinline__ double4 at(uint32_t n) const {
    if constexpr (VIEW == kMcRecords) return pos[n];
    // n / ny: magic is 2^32 / ny less at most 1, and n < 2^31, so the product's
    // high word is the quotient or one less
    uint32_t i = __umulhi(n, magic), j = n - i * ny;
    const bool next = j >= ny;
    i += next ? 1u : 0u;
    j -= next ? ny : 0u;
    const double* pw = reinterpret_cast<const double*>(lat.wc + n);
    if constexpr (VIEW == kMcStaged)
      return make_double4(table[ny - row0 + i], table[j], z, *pw);
    const double* px = lat.xy + (kLatticeMaxRow + 1 + i);
    const double* py = lat.xy + j;
    if constexpr (VIEW == kMcTables) return make_double4(*px, *py, z, *pw);
    const bool tab = n < body;
    const double* rec = &pos[n].x;
    px = tab ? px : rec;
    py = tab ? py : rec + 1;
    const double* pz = tab ? lat.xy + kLatticeMaxRow : rec + 2;
    pw = tab ? pw : rec + 3;
    return make_double4(*px, *py, *pz, *pw);
  }
};

// f(view) with the sources' McView, which is uniform.
template <bool FP64, typename F>
__device__ __forceinline__ void with_view(const McSourceView& s, uint32_t N, F&& f) {
  if (FP64 || s.body == 0)
    f(std::integral_constant<McView, kMcRecords>{});
  else if (s.table)
    f(std::integral_constant<McView, kMcStaged>{});
  else if (s.body == N)
    f(std::integral_constant<McView, kMcTables>{});
  else
    f(std::integral_constant<McView, kMcMixed>{});
}

// Per-target estimator; thread i evaluates the target at v[i], whose index
// (the Philox counter) is tmap[i], or i without a map.  Block row blockIdx.y
// takes the draws k in [blockIdx.y kchunk, +kchunk) (kchunk even) of the K and
// writes its share to y[blockIdx.y M + i].
template <int SIGN, bool FP64, bool OBL, bool SHARED_IDX>
__global__ __launch_bounds__(kBlock) void k_mc(
    const double4* __restrict__ pos, const double* __restrict__ ph,
    uint32_t N, const double* __restrict__ v, uint32_t M, const uint32_t* __restrict__ tmap,
    uint32_t K, uint32_t kchunk, uint32_t seed_lo, uint32_t seed_hi, double Kw,
    double inv_lambda, double scale, McLattice lat, int stage, int staged_only,
    double2* __restrict__ y) {
  __shared__ double s_tab[FP64 ? 1 : kMcTable];
  McSourceView source(pos, lat, FP64, N);
  if constexpr (!FP64) {
    const bool staged = source.stages(N);  // uniform
    if (staged_only && !staged) return;
    if (stage && lat.use && staged) source.stage(0, N, s_tab);
  }
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= M) return;
  McDraws d = mc_split(K, kchunk, blockIdx.y);
  const uint32_t m = tmap ? tmap[i] : i;
  const double vx = v[3 * (size_t)i], vy = v[3 * (size_t)i + 1],
               vz = v[3 * (size_t)i + 2];
  double ar = 0.0, ai = 0.0;
  with_view<FP64>(source, N, [&](auto view) {
    float fr = 0.f, fi = 0.f;
    // 8 samples per step: 4 Philox blocks, then 8 independent gathers in flight
    for (; d.left >= 8; d.take(8)) {
      uint32_t idx[8];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const U4 o = mc_draws<SHARED_IDX>(d.k + 2 * h, m, seed_lo, seed_hi);
        idx[2 * h] = lemire_index(o.x, o.y, N);
        idx[2 * h + 1] = lemire_index(o.z, o.w, N);
      }
      double4 p[8];
      double phv[8];
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        p[h] = source.at<view.value>(idx[h]);
        if constexpr (FP64) phv[h] = ph[idx[h]];
      }
      __builtin_amdgcn_sched_barrier(0);  // all loads before the first pair
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        if constexpr (FP64) {
          const PairF64 q =
              pair_f64<SIGN, 0, OBL>(p[h].w, phv[h], p[h].x, p[h].y, p[h].z, vx, vy, vz, Kw);
          accumulate_phasor<0>(q.r, q.arg, ar, ai);
        } else {
          mc_pair_f32s<SIGN, OBL>(p[h], vx, vy, vz, inv_lambda, fr, fi);
        }
      }
      if constexpr (!FP64) {
        ar += fr;
        ai += fi;
        fr = 0.f;
        fi = 0.f;
      }
    }
    for (; d.left; d.take(2)) {
      const U4 o = mc_draws<SHARED_IDX>(d.k, m, seed_lo, seed_hi);
      const uint32_t idx[2] = {lemire_index(o.x, o.y, N), lemire_index(o.z, o.w, N)};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h == 1 && d.left == 1) break;
        const double4 p = source.at<view.value>(idx[h]);
        if constexpr (FP64) {
          const PairF64 q = pair_f64<SIGN, 0, OBL>(p.w, ph[idx[h]], p.x, p.y, p.z, vx, vy, vz, Kw);
          accumulate_phasor<0>(q.r, q.arg, ar, ai);
        } else {
          mc_pair_f32s<SIGN, OBL>(p, vx, vy, vz, inv_lambda, fr, fi);
        }
      }
    }
    ar += fr;
    ai += fi;
  });
  y[(size_t)blockIdx.y * M + i] = make_double2(ar * scale, ai * scale);
}

// Per-target Monte Carlo over source ranges.  A per-target draw gathers one
// random source; from a 1024^2 plane the gathered data (8 MB of weights on a
// lattice, 32 MB of records otherwise) does not fit the 4 MB L2 of an XCD, and
// the misses bound k_mc.  k_mc_pass takes only the draws whose source index
// lies in a range whose data fits one L2, range after range: each regenerates its
// targets' Philox streams (the indices are k_mc's), queues each lane's in-range
// draws in that lane's LDS ring and evaluates them 8 at a time, every lane of the
// wave taking 8 once each active lane holds 8; a ring that could overflow in the
// next round forces a partial batch (lanes with fewer entries idle in it).  A
// launch takes the ranges [b0, b1) and adds their sums into y[m] (FP64): the first
// writes, the last scales by N / K.  The summation order of a target is fixed by
// its indices and the ranges.
// What bounds it: the lines that the L2s deliver, one of 128 bytes for each draw's
// weight (32.6 TB/s; 34 where everything hits), which is why the other two gathers,
// from the row and column tables, are staged in LDS (STAGE: they fit kMcTable
// entries, three workgroups to a CU): as L1 gathers they kept the address units
// busy at 55 cycles each.  1024^2 lattice to 1024^2 targets, K = 1024: 5.3 -> 4.26 ms.
// Idle slots read source lo, one line for all (their old entries: 4.78 ms).  Weights
// loaded past the caches (nontemporal): 11.9 ms.  Records (jittered): 14.3 -> 7.6 ms.
constexpr uint32_t kMcQueue = 32;  // ring slots per lane, a power of two

template <McView VIEW, int SIGN, bool FP64, bool OBL>
__device__ __forceinline__ void mc_pass(const McSourceView& source, const double* __restrict__ ph,
                                        uint32_t N, double vx, double vy, double vz, bool active,
                                        uint32_t m, McDraws d, uint32_t seed_lo, uint32_t seed_hi,
                                        double Kw, double inv_lambda,
                                        uint32_t lo, uint32_t hi, uint32_t* s_q, double& ar,
                                        double& ai) {
  // byte offsets into the ring [slot][lane]: one bank per lane
  constexpr uint32_t kStep = kBlock * sizeof(uint32_t), kMask = (kMcQueue - 1) * kStep;
  const uint32_t t = threadIdx.x * (uint32_t)sizeof(uint32_t);
  const auto slot = [&](uint32_t at) __attribute__((always_inline)) -> uint32_t& {
    return *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(s_q) + ((at & kMask) | t));
  };
  uint32_t head = 0, tail = 0;
  // the next 8 queued draws of every lane, or up to 8; idle lanes drop their terms by
  // a select (never multiplied by zero: a target at source lo would turn 0 * inf
  // into NaN)
  const auto batch = [&](auto full) __attribute__((always_inline)) {
    const uint32_t take = full.value ? 8 * kStep : min(8 * kStep, tail - head);
    uint32_t idx[8];
#pragma unroll
    for (uint32_t h = 0; h < 8; ++h) {
      const uint32_t n = slot(head + h * kStep);
      idx[h] = active && h * kStep < take ? n : lo;  // idle slots all read one line
    }
    double4 p[8];
    double phv[8];
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      p[h] = source.template at<VIEW>(idx[h]);
      if constexpr (FP64) phv[h] = ph[idx[h]];
    }
    __builtin_amdgcn_sched_barrier(0);  // all loads before the first pair
    float fr[2] = {0.f, 0.f}, fi[2] = {0.f, 0.f};  // sums of four in FP32
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      const bool use = full.value || h * kStep < take;
      if constexpr (FP64) {
        const PairF64 q =
            pair_f64<SIGN, 0, OBL>(p[h].w, phv[h], p[h].x, p[h].y, p[h].z, vx, vy, vz, Kw);
        double tr = 0.0, ti = 0.0;
        accumulate_phasor<0>(q.r, q.arg, tr, ti);
        ar += use ? tr : 0.0;
        ai += use ? ti : 0.0;
      } else {
        float tr = fr[h / 4], ti = fi[h / 4];
        mc_pair_f32s<SIGN, OBL>(p[h], vx, vy, vz, inv_lambda, tr, ti);
        fr[h / 4] = use ? tr : fr[h / 4];
        fi[h / 4] = use ? ti : fi[h / 4];
      }
    }
    if constexpr (!FP64) {
      ar += (double)fr[0] + (double)fr[1];
      ai += (double)fi[0] + (double)fi[1];
    }
    head += take;
  };
  for (;; d.take(8)) {
    const bool more = d.left != 0;
    if (more) {
      uint32_t idx[8];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const U4 o = mc_draws<false>(d.k + 2 * h, m, seed_lo, seed_hi);
        idx[2 * h] = lemire_index(o.x, o.y, N);
        idx[2 * h + 1] = lemire_index(o.z, o.w, N);
      }
      const uint32_t width = active ? hi - lo : 0u;
#pragma unroll
      for (uint32_t h = 0; h < 8; ++h)
        if (h < d.left && idx[h] - lo < width) {
          slot(tail) = idx[h];
          tail += kStep;
        }
      // full batches while every active lane holds 8 (idle lanes count as full)
      while (__builtin_amdgcn_ballot_w64(active && tail - head < 8 * kStep) == 0)
        batch(std::true_type{});
    }
    // every ring holds at most kMcQueue - 8 entries before the next round, none
    // after the last
    while (__builtin_amdgcn_ballot_w64(
               active && tail - head > (more ? (kMcQueue - 8) * kStep : 0u)) != 0)
      batch(std::false_type{});
    if (!more) break;
  }
}

template <bool STAGE, int SIGN, bool FP64, bool OBL>
__global__ __launch_bounds__(kBlock) void k_mc_pass(
    const double4* __restrict__ pos, const double* __restrict__ ph, uint32_t N,
    const double* __restrict__ v, uint32_t M, uint32_t K, uint32_t kchunk, uint32_t seed_lo,
    uint32_t seed_hi, double Kw, double inv_lambda, McLattice lat, uint32_t b0, uint32_t b1,
    uint32_t passes,
    uint32_t widest, int staged, double scale, double2* __restrict__ y) {
  __shared__ uint32_t s_q[kMcQueue * kBlock];
  // (without the tables five workgroups' rings fill a CU's LDS)
  double* s_tab = nullptr;
  if constexpr (STAGE) {
    __shared__ double tab[kMcTable];
    s_tab = tab;
  }
  McSourceView source(pos, lat, FP64, N);
  if (widest && source.stages(widest) != (staged != 0)) return;  // uniform
  const uint32_t m = blockIdx.x * kBlock + threadIdx.x;
  const bool active = m < M, idle = __ballot(active) == 0;  // idle: the whole wave is past M
  const uint32_t mm = active ? m : M - 1;
  const double vx = v[3 * (size_t)mm], vy = v[3 * (size_t)mm + 1], vz = v[3 * (size_t)mm + 2];
  const McDraws draws = mc_split(K, kchunk, blockIdx.y);
  y += (size_t)blockIdx.y * M;
  double ar = 0.0, ai = 0.0;
  for (uint32_t b = b0; b < b1; ++b) {
    const uint32_t lo = (uint32_t)((uint64_t)b * N / passes);
    const uint32_t hi = (uint32_t)((uint64_t)(b + 1) * N / passes);
    if constexpr (STAGE) {
      __syncthreads();  // the previous range's reads are done
      source.stage(lo, hi, s_tab);
    }
    if (idle) continue;
    const auto run = [&](auto view) __attribute__((always_inline)) {
      mc_pass<view.value, SIGN, FP64, OBL>(source, ph, N, vx, vy, vz, active, mm, draws, seed_lo,
                                           seed_hi, Kw, inv_lambda, lo, hi, s_q, ar, ai);
    };
    if constexpr (STAGE)
      run(std::integral_constant<McView, kMcStaged>{});
    else
      with_view<FP64>(source, N, run);
  }
  if (active) {
    if (b0) {
      const double2 old = y[m];
      ar += old.x;
      ai += old.y;
    }
    if (b1 < passes) scale = 1.0;
    y[m] = make_double2(ar * scale, ai * scale);
  }
}

// Batched Monte Carlo: one workgroup = one group of kMcGroup targets
// (kBlock lanes x 4 targets each) sharing the subset n_{g,k}.
template <int SIGN, bool FP64, bool OBL>
__global__ __launch_bounds__(kBlock) void k_mc_shared(
    const double4* __restrict__ pos, const double* __restrict__ ph,
    uint32_t N, const double* __restrict__ v, uint32_t M, uint32_t K, uint32_t kchunk,
    uint32_t seed_lo, uint32_t seed_hi, double Kw, double inv_lambda,
    double scale, double2* __restrict__ y) {
  constexpr int R = kMcGroup / kBlock;
  McDraws d = mc_split(K, kchunk, blockIdx.y);  // kchunk: of 64
  y += (size_t)blockIdx.y * M;
  const uint32_t g = blockIdx.x;
  double vx[R], vy[R], vz[R], ar[R], ai[R];
  float fr[R], fi[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t m = g * kMcGroup + r * kBlock + threadIdx.x;
    const size_t mm = m < M ? m : M - 1;
    vx[r] = v[3 * mm];
    vy[r] = v[3 * mm + 1];
    vz[r] = v[3 * mm + 2];
    ar[r] = ai[r] = 0.0;
    fr[r] = fi[r] = 0.f;
  }
  for (; d.left; d.take(2)) {
    const U4 o = philox4x32_10(U4{d.k >> 1, g, kMcSharedTag, kMcStream}, seed_lo, seed_hi);
    const uint32_t idx[2] = {lemire_index(o.x, o.y, N), lemire_index(o.z, o.w, N)};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h == 1 && d.left == 1) break;
      const double4 p = pos[idx[h]];
      if constexpr (FP64) {
        const double phv = ph[idx[h]];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const PairF64 q =
              pair_f64<SIGN, 0, OBL>(p.w, phv, p.x, p.y, p.z, vx[r], vy[r], vz[r], Kw);
          accumulate_phasor<0>(q.r, q.arg, ar[r], ai[r]);
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
          mc_pair_f32s<SIGN, OBL>(p, vx[r], vy[r], vz[r], inv_lambda, fr[r], fi[r]);
      }
    }
    if constexpr (!FP64) {
      if ((d.k & 62) == 62 || d.left <= 2) {  // flush FP32 partials every 64 draws
#pragma unroll
        for (int r = 0; r < R; ++r) {
          ar[r] += fr[r];
          ai[r] += fi[r];
          fr[r] = fi[r] = 0.f;
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t m = g * kMcGroup + r * kBlock + threadIdx.x;
    if (m < M) y[m] = make_double2(ar[r] * scale, ai[r] * scale);
  }
}

// Ranges of about `per_pass` bytes over `bytes` gathered, at most `most` (option
// "mc_passes" sets the number).
static uint32_t mc_passes(size_t N, size_t bytes, size_t per_pass, size_t most = 8) {
  const int opt = tuning().mc_passes;
  if (opt > 0) return (uint32_t)std::min<size_t>((size_t)opt, std::max<size_t>(N, 1));
  const size_t p = (bytes + per_pass - 1) / per_pass;
  return (uint32_t)std::min<size_t>(std::max<size_t>(p, 1), most);
}

static bool mc_round(size_t blocks, bool fp64) {
  return blocks <= (fp64 ? kMcRound / 3 : kMcRound);
}

uint32_t mc_splits(size_t M, uint32_t K, bool fp64, bool shared, size_t cap,
                   uint32_t* chunk) {
  const size_t group = shared ? kMcGroup : (size_t)kBlock, blocks = (M + group - 1) / group;
  const size_t fill = shared ? 2048 : kMcRound, least = shared ? 64 : kMcMinDraws;
  size_t S = std::min<size_t>({fill / blocks, K / least, 64});
  if (!shared && !mc_round(blocks, fp64)) S = 1;  // ranges add to y launch by launch
  S = std::min(S, cap / M);
  return mc_chunk(K, S, shared ? 64 : 8, chunk);
}

hipError_t launch_mc(int sign, bool fp64, bool shared, bool obliquity, const double4* pos,
                     const double* ph, size_t N, const double* v, size_t M,
                     uint32_t K, uint64_t seed, double K_wave, double lambda,
                     const McLattice& lat, double2* y, double2* partial,
                     size_t partial_cap, hipStream_t stream) {
  if (!M) return hipSuccess;
  const double scale = (double)N / (double)K;
  const uint32_t slo = (uint32_t)seed, shi = (uint32_t)(seed >> 32);
  const double il = 1.0 / lambda;
  const unsigned blocks = shared ? (unsigned)((M + kMcGroup - 1) / kMcGroup)
                                 : (unsigned)((M + kBlock - 1) / kBlock);
  uint32_t chunk;
  const uint32_t S = mc_splits(M, K, fp64, shared, partial_cap, &chunk);
  double2* out = S > 1 ? partial : y;
  const dim3 grid(blocks, S);
  const bool round = mc_round(blocks, fp64);
  const uint64_t draws = (uint64_t)M * K;
  // FP64 gathers 40 bytes per draw.  FP32-split sources gather 8 on a lattice; off it
  // 32, which take ranges of their own where the draws pay for them.
  const size_t mb = size_t(1) << 20;
  uint32_t passes;
  if (fp64)
    passes = mc_passes(N, 40 * N, 3 * mb, round ? 3 : 8);
  else if (!round && draws >= kMcRecordDraws)
    passes = mc_passes(N, 32 * N, 4 * mb);
  else
    passes = mc_passes(N, 8 * N, 3 * mb);
  const bool apart = !fp64 && lat.info && passes > 1 &&
                     draws >= (round ? kMcStageDraws / 8 : kMcStageDraws);
  with_sign(sign, [&](auto sg) {
    with_bool(fp64, [&](auto f64) {
      with_bool(obliquity, [&](auto obl) {
        if (shared) {
          k_mc_shared<sg.value, (bool)f64.value, (bool)obl.value><<<grid, kBlock, 0, stream>>>(
              pos, ph, (uint32_t)N, v, (uint32_t)M, K, chunk, slo, shi, K_wave, il, scale, out);
          return;
        }
        // widest: 0, or the width of the staged ranges, and the launch is for the
        // sources that can (`staged`) or cannot be staged and exits on the others
        const auto ranges = [&](auto stage, uint32_t passes, uint32_t widest, bool staged) {
          if (passes <= 1)
            k_mc<sg.value, (bool)f64.value, (bool)obl.value, false><<<grid, kBlock, 0, stream>>>(
                pos, ph, (uint32_t)N, v, (uint32_t)M, nullptr, K, chunk, slo, shi, K_wave, il,
                scale, lat, chunk >= kMcStageK ? 1 : 0, widest ? 1 : 0, out);
          else
            for (uint32_t b = 0; b < passes; b = round ? passes : b + 1)
              k_mc_pass<(bool)stage.value, sg.value, (bool)f64.value, (bool)obl.value>
                  <<<grid, kBlock, 0, stream>>>(pos, ph, (uint32_t)N, v, (uint32_t)M, K, chunk,
                                                slo, shi, K_wave, il, lat, b,
                                                round ? passes : b + 1, passes, widest,
                                                staged ? 1 : 0, scale, out);
        };
        if constexpr (!(bool)f64.value) {
          if (apart) {
            const uint32_t staged = mc_passes(N, 8 * N, 4 * mb);
            const uint32_t widest = (uint32_t)((N + staged - 1) / staged);
            if (lat.use)
              ranges(std::true_type{}, staged, widest, true);
            else
              ranges(std::false_type{}, staged, widest, true);
            ranges(std::false_type{}, passes, widest, false);
            return;
          }
        }
        ranges(std::false_type{}, passes, 0u, false);
      });
    });
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_reduce_partials((int)S, M, partial, y, stream);
}

hipError_t launch_mc_subset(int sign, bool shared, bool obliquity, const double4* pos,
                            const double* ph, size_t N, const double* vsub, size_t count,
                            const uint32_t* tmap, uint32_t K, uint64_t seed, double K_wave,
                            double lambda, double2* y, double2* partial, size_t partial_cap,
                            hipStream_t stream) {
  if (!count) return hipSuccess;
  const double scale = (double)N / (double)K;
  const uint32_t slo = (uint32_t)seed, shi = (uint32_t)(seed >> 32);
  const unsigned blocks = (unsigned)((count + kBlock - 1) / kBlock);
  // a few hundred targets: the draws are split into chunks of at least 64
  // (a multiple of 8) over enough blocks to fill the GPU, summed in order
  uint32_t chunk;
  const uint32_t S = mc_chunk(
      K, std::min<size_t>({((size_t)K + 63) / 64, kFewTargetSplits, partial_cap / count}), 8,
      &chunk);
  double2* out = S > 1 ? partial : y;
  with_sign(sign, [&](auto sg) {
    with_bool(shared, [&](auto sh) {
      with_bool(obliquity, [&](auto obl) {
        k_mc<sg.value, true, (bool)obl.value, (bool)sh.value>
            <<<dim3(blocks, S), kBlock, 0, stream>>>(pos, ph, (uint32_t)N, vsub,
                                                     (uint32_t)count, tmap, K, chunk, slo, shi,
                                                     K_wave, 1.0 / lambda, scale, McLattice{},
                                                     0, 0, out);
      });
    });
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_reduce_partials((int)S, count, partial, y, stream);
}

__global__ __launch_bounds__(kBlock) void k_mc_pack(
    int fp64, const double* __restrict__ amp, const double* __restrict__ phase,
    const double* __restrict__ u, uint32_t N, double4* __restrict__ pos,
    double* __restrict__ ph, float2* __restrict__ wc) {
  const uint32_t n = blockIdx.x * kBlock + threadIdx.x;
  if (n >= N) return;
  double4 p;
  p.x = u[3 * (size_t)n];
  p.y = u[3 * (size_t)n + 1];
  p.z = u[3 * (size_t)n + 2];
  if (fp64) {
    p.w = amp[n];
    ph[n] = phase[n];
  } else {
    double sn, cs;
    sincos(phase[n], &sn, &cs);
    const float2 w = make_float2((float)(amp[n] * cs), (float)(amp[n] * sn));
    p.w = __builtin_bit_cast(double, w);
    if (wc) wc[n] = w;
  }
  pos[n] = p;
}

hipError_t launch_mc_pack(bool fp64, const double* amp, const double* phase,
                          const double* u, size_t N, double4* pos, double* ph, float2* wc,
                          hipStream_t stream) {
  if (!N) return hipSuccess;
  const unsigned blocks = (unsigned)((N + kBlock - 1) / kBlock);
  k_mc_pack<<<blocks, kBlock, 0, stream>>>(fp64 ? 1 : 0, amp, phase, u,
                                          (uint32_t)N, pos, ph, wc);
  return hipGetLastError();
}

// Row length of an x-slow product grid: the first n with x_n != x_0, among
// n < min(N, kLatticeMaxRow); N when all x are equal and N <= kLatticeMaxRow;
// 0 (not a grid) otherwise.  info[0] = that length ny, info[1] = N / ny, the
// number of whole rows, which k_lattice_check lowers to the number of leading
// complete rows.
__global__ __launch_bounds__(kBlock) void k_lattice_row(const double* __restrict__ u,
                                                        uint32_t N, uint32_t* __restrict__ info) {
  __shared__ uint32_t s_min[kBlock / 64];
  const double x0 = u[0];
  const uint32_t lim = min(N, kLatticeMaxRow);
  uint32_t first = lim;
  for (uint32_t n = 1 + threadIdx.x; n < lim; n += kBlock)
    if (u[3 * (size_t)n] != x0) {  // this thread's first hit is its smallest
      first = n;
      break;
    }
  for (int off = 32; off; off >>= 1) first = min(first, (uint32_t)__shfl_xor((int)first, off, 64));
  if ((threadIdx.x & 63) == 0) s_min[threadIdx.x >> 6] = first;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t f = lim;
    for (int w = 0; w < kBlock / 64; ++w) f = min(f, s_min[w]);
    const uint32_t ny = f < lim ? f : (N <= kLatticeMaxRow ? N : 0u);
    info[0] = ny;
    info[1] = ny ? N / ny : 0u;
  }
}

// Checks u[n] == (x of row n / ny, y of column n % ny, z_0) exactly for the
// sources of the whole rows and lowers info[1] to the first row where it fails
// (an atomic minimum: order-free), so that info[1] rows lead complete (a
// padded plane's copies of source 0 repeat row 0's y and never complete a
// row); fills the tables described with McLattice.
__global__ __launch_bounds__(kBlock) void k_lattice_check(const double* __restrict__ u,
                                                          uint32_t N, uint32_t* __restrict__ info,
                                                          double* __restrict__ xy) {
  const uint32_t ny = info[0];
  const uint32_t n = blockIdx.x * kBlock + threadIdx.x;
  if (!ny || n >= (N / ny) * ny) return;
  const uint32_t i = n / ny, j = n - i * ny;
  const double x = u[3 * (size_t)n], y = u[3 * (size_t)n + 1], z = u[3 * (size_t)n + 2];
  if (!(x == u[3 * (size_t)i * ny] && y == u[3 * (size_t)j + 1] && z == u[2]))
    atomicMin(&info[1], i);
  if (j == 0) xy[kLatticeMaxRow + 1 + i] = x;
  if (i == 0) xy[j] = y;
  if (n == 0) xy[kLatticeMaxRow] = z;
}

hipError_t launch_mc_lattice_probe(const double* u, size_t N, uint32_t* info, double* xy,
                                   hipStream_t stream) {
  if (!N) return hipSuccess;
  k_lattice_row<<<1, kBlock, 0, stream>>>(u, (uint32_t)N, info);
  const unsigned blocks = (unsigned)((N + kBlock - 1) / kBlock);
  k_lattice_check<<<blocks, kBlock, 0, stream>>>(u, (uint32_t)N, info, xy);
  return hipGetLastError();
}

__global__ __launch_bounds__(kBlock) void k_mc_indices(
    uint32_t seed_lo, uint32_t seed_hi, uint64_t N, uint32_t m0,
    uint32_t count, uint32_t K, uint32_t tag, int64_t* __restrict__ idx) {
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j >= count) return;
  const uint32_t m = m0 + j;
  for (McDraws d{0u, K}; d.left; d.take(2)) {
    const uint32_t k = d.k;
    const U4 o = philox4x32_10<true>(U4{k >> 1, m, tag, kMcStream}, seed_lo, seed_hi);
    idx[(size_t)j * K + k] = lemire_index(o.x, o.y, (uint32_t)N);
    if (d.left > 1) idx[(size_t)j * K + k + 1] = lemire_index(o.z, o.w, (uint32_t)N);
  }
}

hipError_t launch_mc_indices(uint64_t seed, uint64_t N, size_t m0,
                             size_t count, uint32_t K, bool shared, int64_t* idx,
                             hipStream_t stream) {
  if (!count || !K) return hipSuccess;
  const unsigned blocks = (unsigned)((count + kBlock - 1) / kBlock);
  k_mc_indices<<<blocks, kBlock, 0, stream>>>((uint32_t)seed,
                                             (uint32_t)(seed >> 32), N,
                                             (uint32_t)m0, (uint32_t)count, K,
                                             shared ? kMcSharedTag : 0u, idx);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// time_transform post-processing (cuda/transform.cu:106-139, 400-405):
// max |y| (order-free, so deterministic), then polar(y / max).

constexpr unsigned kMaxBlocks = 1024;

__device__ __forceinline__ double wave_max(double x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = fmax(x, __shfl_xor(x, off));
  return x;
}

__global__ __launch_bounds__(kBlock) void k_max_abs(
    const double2* __restrict__ y, uint32_t M, double* __restrict__ block_max) {
  __shared__ double red[kBlock / 64];
  double mx = 0.0;
  for (uint32_t m = blockIdx.x * kBlock + threadIdx.x; m < M;
       m += gridDim.x * kBlock) {
    const double2 z = y[m];
    mx = fmax(mx, hypot(z.x, z.y));
  }
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    double b = red[0];
    for (int i = 1; i < kBlock / 64; ++i) b = fmax(b, red[i]);
    block_max[blockIdx.x] = b;
  }
}

__global__ __launch_bounds__(kBlock) void k_final_max(
    const double* __restrict__ block_max, uint32_t nb,
    double* __restrict__ max_out) {
  __shared__ double red[kBlock / 64];
  double mx = 0.0;
  for (uint32_t i = threadIdx.x; i < nb; i += kBlock) mx = fmax(mx, block_max[i]);
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    double b = red[0];
    for (int i = 1; i < kBlock / 64; ++i) b = fmax(b, red[i]);
    max_out[0] = b;
  }
}

__global__ __launch_bounds__(kBlock) void k_to_polar(
    const double2* __restrict__ y, uint32_t M,
    const double* __restrict__ max_in, double* __restrict__ amp,
    double* __restrict__ phase) {
  const uint32_t m = blockIdx.x * kBlock + threadIdx.x;
  if (m >= M) return;
  const double mx = max_in[0];
  const double div = mx < 1e-6 ? 1.0 : mx;
  const double2 z = y[m];
  const double re = z.x / div, im = z.y / div;
  amp[m] = hypot(re, im);
  phase[m] = atan2(im, re);
}

hipError_t launch_normalize_polar(const double2* y, size_t M, double* amp,
                                  double* phase, double* max_out,
                                  double* scratch, hipStream_t stream) {
  if (!M) return hipSuccess;
  unsigned nb = (unsigned)std::min<size_t>((M + kBlock - 1) / kBlock, kMaxBlocks);
  k_max_abs<<<nb, kBlock, 0, stream>>>(y, (uint32_t)M, scratch);
  k_final_max<<<1, kBlock, 0, stream>>>(scratch, nb, max_out);
  const unsigned blocks = (unsigned)((M + kBlock - 1) / kBlock);
  k_to_polar<<<blocks, kBlock, 0, stream>>>(y, (uint32_t)M, max_out, amp, phase);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Error report of an FP32-split result y (M values), from count FP64 values
// at sampled targets: n_e of them drawn by the result's energy and n_u
// spread evenly (multiple importance sampling with the balance heuristic).
// Energy draw i < n_e is the target at which the running sum of |y|^2 in
// target order first exceeds (i + 1/2) / n_e of the total T; even draw j is
// target floor(j M / n_u).  Then
//   err^2 = sum_i |y[m_i] - ref_i|^2 / (n_e |y[m_i]|^2 + n_u T / M),
// an unbiased estimate (under random offsets of the strata) of
// sum_m |y_m - y64_m|^2 / T, the whole result's squared relative L2 error:
// the energy draws find error that grows with the field (a focus), the even
// ones error spread over dark targets.  M <= count takes every target once
// (n_e = 0: the exact value).  A result without a finite positive T takes
// the even targets and sqrt(sum |y - ref|^2 / sum |ref|^2) there.  Every sum
// has a fixed order.

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

// inclusive prefix sum over the 64 lanes (a fixed order)
__device__ __forceinline__ double wave_scan(double x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double t = __shfl_up(x, off);
    if (lane >= off) x += t;
  }
  return x;
}

__device__ __forceinline__ double energy(const double2 a) { return a.x * a.x + a.y * a.y; }

// sum of E[0 .. n) by one wave, the same bits wherever it is called
__device__ __forceinline__ double energy_total(const double* __restrict__ E, uint32_t n) {
  double s = 0.0;
  for (uint32_t b = threadIdx.x & 63; b < n; b += 64) s += E[b];
  return wave_sum(s);
}

__device__ __forceinline__ bool energy_mode(double total) {
  return total > 0.0 && __builtin_isfinite(total);  // NaN fails
}

// Block b: E[b] = sum of |y|^2 over its chunk [b L, min(M, (b + 1) L)).
__global__ __launch_bounds__(kBlock) void k_energy_chunks(const double2* __restrict__ y,
                                                          uint32_t M, uint32_t L,
                                                          double* __restrict__ E) {
  __shared__ double red[kBlock / 64];
  const uint64_t b0 = (uint64_t)blockIdx.x * L, b1 = min<uint64_t>(M, b0 + L);
  double s = 0.0;
  for (uint64_t m = b0 + threadIdx.x; m < b1; m += kBlock) s += energy(y[m]);
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) t += red[w];
    E[blockIdx.x] = t;
  }
}

// One wave per sample i: m_i as above, into tmap[i] and its position into vsub.
__global__ __launch_bounds__(kBlock) void k_error_targets(
    const double2* __restrict__ y, uint32_t M, uint32_t L, const double* __restrict__ E,
    uint32_t nchunks, const double* __restrict__ v, uint32_t count, uint32_t ne,
    uint32_t* __restrict__ tmap, double* __restrict__ vsub) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (i >= count) return;  // the whole wave
  const double total = energy_total(E, nchunks);
  const bool draw = energy_mode(total) && i < ne;
  const uint32_t j = energy_mode(total) ? i - ne : i, nu = energy_mode(total) ? count - ne : count;
  uint32_t m = draw ? 0u : (uint32_t)(((uint64_t)j * M) / nu);
  if (draw) {
    const double c = ((double)i + 0.5) / (double)ne * total;
    // the chunk where the running sum passes c (else the last one with energy)
    uint32_t cb = nchunks, lastb = nchunks;
    double before = 0.0, lastbefore = 0.0, run = 0.0;
    for (uint32_t base = 0; base < nchunks && cb == nchunks; base += 64) {
      const double e = base + lane < nchunks ? E[base + lane] : 0.0;
      const double incl = wave_scan(e) + run;
      const uint64_t hit = __ballot(incl > c && e > 0.0);
      const uint64_t pos = __ballot(e > 0.0);
      if (hit) {
        const uint32_t f = (uint32_t)__builtin_ctzll(hit);
        cb = base + f;
        before = __shfl(incl - e, f);
      } else if (pos) {
        const uint32_t f = 63u - (uint32_t)__builtin_clzll(pos);
        lastb = base + f;
        lastbefore = __shfl(incl - e, f);
      }
      run = __shfl(incl, 63);
    }
    if (cb == nchunks) {
      cb = lastb;
      before = lastbefore;
    }
    // within the chunk, likewise (else its last target with energy)
    const uint64_t b0 = (uint64_t)cb * L, b1 = min<uint64_t>(M, b0 + L);
    uint64_t found = b1, last = b0;
    run = before;
    for (uint64_t base = b0; base < b1 && found == b1; base += 64) {
      const double e = base + lane < b1 ? energy(y[base + lane]) : 0.0;
      const double incl = wave_scan(e) + run;
      const uint64_t hit = __ballot(incl > c && e > 0.0);
      const uint64_t pos = __ballot(e > 0.0);
      if (hit) found = base + (uint64_t)__builtin_ctzll(hit);
      else if (pos) last = base + 63u - (uint64_t)__builtin_clzll(pos);
      run = __shfl(incl, 63);
    }
    m = (uint32_t)(found < b1 ? found : last);
  }
  if (lane == 0) {
    tmap[i] = m;
    vsub[3 * (size_t)i] = v[3 * (size_t)m];
    vsub[3 * (size_t)i + 1] = v[3 * (size_t)m + 1];
    vsub[3 * (size_t)i + 2] = v[3 * (size_t)m + 2];
  }
}

uint32_t error_chunk_len(size_t M) {
  return (uint32_t)std::max<size_t>((M + kErrChunks - 1) / kErrChunks, 1);
}

uint32_t error_energy_draws(size_t M, size_t count) {
  return M <= count ? 0u : (uint32_t)(count / 2);
}

hipError_t launch_error_targets(const double2* y, size_t M, const double* v, size_t count,
                                double* E, uint32_t* tmap, double* vsub, hipStream_t stream) {
  if (!count) return hipSuccess;
  const uint32_t L = error_chunk_len(M);
  const uint32_t nchunks = (uint32_t)((M + L - 1) / L);
  k_energy_chunks<<<nchunks, kBlock, 0, stream>>>(y, (uint32_t)M, L, E);
  const unsigned blocks = (unsigned)((count + kBlock / 64 - 1) / (kBlock / 64));
  k_error_targets<<<blocks, kBlock, 0, stream>>>(y, (uint32_t)M, L, E, nchunks, v,
                                                 (uint32_t)count, error_energy_draws(M, count),
                                                 tmap, vsub);
  return hipGetLastError();
}

// One workgroup: the report from the sampled targets (weighted, or the even
// targets alone, as k_error_targets chose from the same E).
__global__ __launch_bounds__(kBlock) void k_rel_l2(const double2* __restrict__ y, uint32_t M,
                                                   const uint32_t* __restrict__ tmap,
                                                   const double2* __restrict__ ref,
                                                   uint32_t count, uint32_t ne,
                                                   const double* __restrict__ E,
                                                   uint32_t nchunks, double* __restrict__ err) {
  __shared__ double red[2][kBlock / 64];
  __shared__ double s_total;
  if (threadIdx.x < 64) {
    const double t = energy_total(E, nchunks);
    if (threadIdx.x == 0) s_total = t;
  }
  __syncthreads();
  const bool weighted = energy_mode(s_total);
  // n_u T / M, the even draws' share of the weight
  const double even = (double)(count - ne) * (s_total / (double)M);
  double num = 0.0, den = 0.0;
  for (uint32_t i = threadIdx.x; i < count; i += kBlock) {
    const double2 a = y[tmap[i]], b = ref[i];
    const double dr = a.x - b.x, di = a.y - b.y;
    if (weighted) {
      num += (dr * dr + di * di) / ((double)ne * energy(a) + even);
    } else {
      num += dr * dr + di * di;
      den += energy(b);
    }
  }
  num = wave_sum(num);
  den = wave_sum(den);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = num;
    red[1][threadIdx.x >> 6] = den;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double n = 0.0, d = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) {
      n += red[0][w];
      d += red[1][w];
    }
    if (weighted) err[0] = __builtin_sqrt(n);
    else err[0] = d > 0.0 ? __builtin_sqrt(n / d) : (n > 0.0 ? INFINITY : 0.0);
  }
}

hipError_t launch_rel_l2(const double2* y, size_t M, const uint32_t* tmap, const double2* ref,
                         size_t count, const double* E, double* err, hipStream_t stream) {
  const uint32_t L = error_chunk_len(M);
  k_rel_l2<<<1, kBlock, 0, stream>>>(y, (uint32_t)M, tmap, ref, (uint32_t)count,
                                     error_energy_draws(M, count), E,
                                     (uint32_t)((M + L - 1) / L), err);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------

// Zero fill with a kernel rather than hipMemsetAsync, so that device-pointer
// calls stay safe to record into a HIP graph.
__global__ __launch_bounds__(kBlock) void k_zero(double* __restrict__ x,
                                                 size_t n) {
  for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n;
       i += (size_t)gridDim.x * kBlock)
    x[i] = 0.0;
}

hipError_t launch_zero(double* x, size_t n, hipStream_t stream) {
  if (!n) return hipSuccess;
  const unsigned blocks = (unsigned)std::min<size_t>((n + kBlock - 1) / kBlock, 4096);
  k_zero<<<blocks, kBlock, 0, stream>>>(x, n);
  return hipGetLastError();
}

__global__ __launch_bounds__(kBlock) void k_adjoint_epilogue(
    const double2* __restrict__ b, const double* __restrict__ amp,
    const double* __restrict__ theta, uint32_t N,
    double* __restrict__ grad_amp, double* __restrict__ grad_theta) {
  const uint32_t n = blockIdx.x * kBlock + threadIdx.x;
  if (n >= N) return;
  double s, c;
  sincos(theta[n], &s, &c);
  const double2 z = b[n];
  const double pr = c * z.x + s * z.y;
  const double pi = c * z.y - s * z.x;
  grad_amp[n] = pr;
  grad_theta[n] = amp[n] * pi;
}

hipError_t launch_adjoint_epilogue(const double2* b, const double* amp,
                                   const double* theta, size_t N,
                                   double* grad_amp, double* grad_theta,
                                   hipStream_t stream) {
  if (!N) return hipSuccess;
  const unsigned blocks = (unsigned)((N + kBlock - 1) / kBlock);
  k_adjoint_epilogue<<<blocks, kBlock, 0, stream>>>(b, amp, theta, (uint32_t)N,
                                                   grad_amp, grad_theta);
  return hipGetLastError();
}

}  // namespace holo
