// A uniform lattice of sources found and tiled on the device, for calls that get
// device positions without a plan: the same decisions and the same bits as the
// plan's host builder (holo_capi.hip: complete_rows, row_length, uniform_z,
// build_grid16), which needs the positions on the host.
//
// What bounds it: latency, three dependent launches of 3 to 4 us, a copy of 64 bytes
// back, and the launch that cuts the tiles; the search reads the positions once, at
// 512^2 sources 6 us.  There the host
// builder took 1.5 ms: 0.6 ms to copy 6.3 MB into fresh pages, the rest to scan and
// cut them, and 0.4 ms to upload the tiles.
#include <hip/hip_runtime.h>
#include <math.h>

#include "holo_device.hpp"
#include "holo_internal.hpp"

namespace holo {

// ny: the first n with x_n != x_0 (0: none below kLatticeFindRow); the other words'
// initial values.
__global__ __launch_bounds__(kBlock) void k_find_row(const double* __restrict__ u, uint32_t N,
                                                     LatticeInfo* __restrict__ info) {
  __shared__ uint32_t s_min[kBlock / 64];
  const double x0 = u[0];
  const uint32_t lim = min(N, kLatticeFindRow);
  uint32_t ny = 0;
  for (uint32_t base = 1; base < lim && !ny; base += 4 * kBlock) {
    uint32_t first = lim;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      const uint32_t n = base + q * kBlock + threadIdx.x;
      if (n < lim && !(u[3 * (size_t)n] == x0)) first = min(first, n);
    }
    for (int off = 32; off; off >>= 1)
      first = min(first, (uint32_t)__shfl_xor((int)first, off, 64));
    if ((threadIdx.x & 63) == 0) s_min[threadIdx.x >> 6] = first;
    __syncthreads();
    for (int w = 0; w < kBlock / 64; ++w) first = min(first, s_min[w]);
    __syncthreads();
    if (first < lim) ny = first;  // uniform
  }
  if (threadIdx.x == 0) {
    info->ny = ny;
    info->rows = ny ? N / ny : 0u;
    info->uniform_z = info->in_rows = info->tail_same = 1u;
    info->uniform = 0u;
  }
}

// The number of leading complete rows, one z for all, one x per run of ny.
__global__ __launch_bounds__(kBlock) void k_find_rows(const double* __restrict__ u, uint32_t N,
                                                      LatticeInfo* __restrict__ info) {
  const uint32_t ny = info->ny, n = blockIdx.x * kBlock + threadIdx.x;
  if (!ny || n >= N) return;
  const uint32_t i = n / ny, j = n - i * ny;
  const double x = u[3 * (size_t)n], y = u[3 * (size_t)n + 1], z = u[3 * (size_t)n + 2];
  const bool same_x = x == u[3 * (size_t)(n - j)], same_z = z == u[2];
  if (!same_z) info->uniform_z = 0u;  // (any number of threads store the same)
  if (!same_x) info->in_rows = 0u;
  if (!(same_x && same_z && y == u[3 * (size_t)j + 1]) && i < N / ny) atomicMin(&info->rows, i);
}

// The pitches of the complete rows, whether they are uniform, and whether the
// sources after the rows are all at one place.
__global__ __launch_bounds__(kBlock) void k_find_pitch(const double* __restrict__ u, uint32_t N,
                                                       LatticeInfo* __restrict__ info) {
#pragma clang fp contract(off)
  const uint32_t ny = info->ny, nx = info->rows;
  if (ny < 2 || nx < 2) return;  // uniform
  const double x0 = u[0], y0 = u[1];
  const double px = (u[3 * (size_t)(nx - 1) * ny] - x0) / (double)(nx - 1);
  const double py = (u[3 * (size_t)(ny - 1) + 1] - y0) / (double)(ny - 1);
  bool ok = px != 0.0 && py != 0.0 && __builtin_isfinite(px) && __builtin_isfinite(py);
  for (uint32_t i = threadIdx.x; i < nx; i += kBlock)
    ok = ok && __builtin_fabs(u[3 * (size_t)i * ny] - (x0 + (double)i * px)) <=
                   1e-9 * __builtin_fabs(px);
  for (uint32_t j = threadIdx.x; j < ny; j += kBlock)
    ok = ok &&
         __builtin_fabs(u[3 * (size_t)j + 1] - (y0 + (double)j * py)) <= 1e-9 * __builtin_fabs(py);
  const uint32_t body = nx * ny;
  bool same = true;
  if (N - body < max(nx, ny))
    for (uint32_t n = body + threadIdx.x; n < N; n += kBlock)
      for (int d = 0; d < 3; ++d)
        same = same && u[3 * (size_t)n + d] == u[3 * (size_t)body + d];
  ok = __syncthreads_and(ok ? 1 : 0) != 0;
  same = __syncthreads_and(same ? 1 : 0) != 0;
  if (threadIdx.x == 0) {
    info->uniform = ok ? 1u : 0u;
    info->tail_same = same ? 1u : 0u;
    info->x0 = x0;
    info->y0 = y0;
    info->z = u[2];
    info->px = px;
    info->py = py;
  }
}

hipError_t launch_find_lattice(const double* u, size_t N, LatticeInfo* info, hipStream_t stream) {
  k_find_row<<<1, kBlock, 0, stream>>>(u, (uint32_t)N, info);
  k_find_rows<<<(unsigned)((N + kBlock - 1) / kBlock), kBlock, 0, stream>>>(u, (uint32_t)N, info);
  k_find_pitch<<<1, kBlock, 0, stream>>>(u, (uint32_t)N, info);
  return hipGetLastError();
}

// The 16-row tiles' slots, centres and axes, as build_grid16 cuts them.
__global__ __launch_bounds__(kBlock) void k_lattice_tiles(LatticeTiles a) {
#pragma clang fp contract(off)
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x, slots = 256 * a.ti * a.tj;
  if (s < slots) {
    const uint32_t t = s >> 8, I = t / a.tj, J = t - I * a.tj;
    const uint32_t i = 16 * I + ((s >> 4) & 15), j = 16 * J + (s & 15);
    a.perm[s] = i < a.nx && j < a.ny ? (int32_t)(i * a.ny + j) : -1;
  } else if (s - slots < a.n_tail) {
    a.perm[s] = (int32_t)(a.nx * a.ny + (s - slots));
  }
  const auto centre = [&](double4* dst, uint32_t cols, uint32_t width, double rho) {
    if (!dst || s >= a.ti * cols) return;
    const uint32_t I = s / cols, J = s - I * cols;
    dst[s] = make_double4(a.x0 + ((double)(16 * I) + 7.5) * a.px,
                          a.y0 + ((double)(width * J) + 0.5 * (double)(width - 1)) * a.py, a.z,
                          rho);
  };
  centre(a.centre16, a.tj, 16, a.rho16);
  centre(a.centre32, a.tj / 2, 32, a.rho32);
  centre(a.centre64, a.tj / 4, 64, a.rho64);
  if (s < 16 * a.ti)
    a.axes[s] = s < a.nx ? a.u[3 * (size_t)s * a.ny] : a.x0 + (double)s * a.px;
  else if (s < 16 * (a.ti + a.tj)) {
    const uint32_t b = s - 16 * a.ti;
    a.axes[s] = b < a.ny ? a.u[3 * (size_t)b + 1] : a.y0 + (double)b * a.py;
  }
}

hipError_t launch_lattice_tiles(const LatticeTiles& a, hipStream_t stream) {
  const size_t n = (size_t)256 * a.ti * a.tj + a.n_tail;
  k_lattice_tiles<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, stream>>>(a);
  return hipGetLastError();
}

}  // namespace holo
