// Host check of the appends' f16 encoder (test harness, built by
// tests/test_oracle.py): any_to_half (csrc/tge_common.h) must give the bits
// of float_to_half_ref for all 2^32 float bit patterns. Prints one JSON line.
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <thread>
#include <vector>

#include "tge_common.h"

int main() {
  const unsigned n = 8;
  std::vector<unsigned long long> wrong(n);
  std::vector<std::thread> threads;
  for (unsigned k = 0; k < n; ++k)
    threads.emplace_back([&, k] {
      unsigned long long w = 0;
      for (uint64_t i = (uint64_t)k << 29; i < (uint64_t)(k + 1) << 29; ++i) {
        const uint32_t u = (uint32_t)i;
        float x;
        memcpy(&x, &u, 4);
        w += tge::any_to_half(x) != tge::float_to_half_ref(x);
      }
      wrong[k] = w;
    });
  unsigned long long w = 0;
  for (unsigned k = 0; k < n; ++k) {
    threads[k].join();
    w += wrong[k];
  }
  printf("{\"mismatches\": %llu}\n", w);
  return w ? 1 : 0;
}
