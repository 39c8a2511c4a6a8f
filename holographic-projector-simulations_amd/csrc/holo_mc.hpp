// How the K draws of a Monte Carlo target split over workgroups and how a split is
// walked, for every K below 2^32: no sum of a draw's index and a step is formed, as
// it would wrap above 2^32 - 8.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#ifdef __HIPCC__
#define HOLO_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define HOLO_HOST_DEVICE inline
#endif

namespace holo {

// The draws k .. k + left - 1 that are still to take.
struct McDraws {
  uint32_t k, left;
  HOLO_HOST_DEVICE void take(uint32_t n) {
    n = left < n ? left : n;
    k += n;
    left -= n;
  }
};

// Split s of the draws, `chunk` to a split (s < mc_chunk's number of splits).
HOLO_HOST_DEVICE McDraws mc_split(uint32_t K, uint32_t chunk, uint32_t s) {
  const uint32_t k = s * chunk, rest = K - k;
  return McDraws{k, rest < chunk ? rest : chunk};
}

// The number of splits, at most `most`, and their draws: a multiple of `step`, or all K.
inline uint32_t mc_chunk(uint32_t K, size_t most, uint32_t step, uint32_t* chunk) {
  const uint64_t S = std::max<uint64_t>(std::min<uint64_t>(most, K), 1);
  const uint64_t c = ((K + S - 1) / S + step - 1) / step * step;
  *chunk = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(c, 1), UINT32_MAX);
  return (uint32_t)(((uint64_t)K + *chunk - 1) / *chunk);
}

}  // namespace holo
