// The splits of K draws (holo_mc.hpp), walked as the kernels walk them: every split
// ends, and together they take each draw once, in order.
#include <cstdio>
#include <cstdlib>

#include "holo_mc.hpp"

int main() {
  using namespace holo;
  const uint64_t top = uint64_t(1) << 32;
  const uint64_t ks[] = {1, 7, 8, 9, 63, 64, 65, 4095, top - 513, top - 512, top - 65, top - 64,
                         top - 63, top - 9, top - 8, top - 7, top - 2, top - 1};
  for (const uint64_t k64 : ks)
    for (const size_t most : {size_t(0), size_t(1), size_t(2), size_t(3), size_t(64), size_t(1024)})
      for (const uint32_t step : {8u, 64u})
        for (const uint32_t walk : {2u, 8u}) {
          const uint32_t K = (uint32_t)k64;
          uint32_t chunk;
          const uint32_t S = mc_chunk(K, most, step, &chunk);
          uint64_t at = 0;
          bool ok = S >= 1 && S <= (most ? most : 1) && (S == 1 || chunk % step == 0);
          for (uint32_t s = 0; s < S; ++s) {
            McDraws d = mc_split(K, chunk, s);
            ok = ok && d.k == at && d.left >= 1;
            at += d.left;
            // the last draws of the split, one by one
            const uint32_t skip = d.left > 100 ? d.left - 100 : 0;
            d.take(skip);
            uint64_t k = d.k;
            int rounds = 0;
            for (; d.left && rounds < 200; d.take(walk), ++rounds) {
              ok = ok && d.k == k;
              k += d.left < walk ? d.left : walk;
            }
            ok = ok && !d.left && k == at;
          }
          if (!ok || at != K) {
            std::printf("K %u, most %zu, step %u: S %u, chunk %u, ends at %llu\n", K, most, step,
                        S, chunk, (unsigned long long)at);
            return 1;
          }
        }
  return 0;
}
