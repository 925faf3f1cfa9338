// Host check of the f16 encoder's branch-free path (test harness, built by
// tests/test_oracle.py): over all 2^32 float bit patterns, a value that
// half_is_normal (csrc/tge_common.h) accepts must encode to the bits of
// float_to_half_ref, and it must accept exactly the magnitudes from 2^-14 up
// to 65536 (exclusive). Prints one JSON line.
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <thread>
#include <vector>

#include "tge_common.h"

int main() {
  const unsigned n = 8;
  std::vector<unsigned long long> accepted(n), wrong(n), range(n);
  std::vector<std::thread> threads;
  for (unsigned k = 0; k < n; ++k)
    threads.emplace_back([&, k] {
      unsigned long long a = 0, w = 0, r = 0;
      for (uint64_t i = (uint64_t)k << 29; i < (uint64_t)(k + 1) << 29; ++i) {
        const uint32_t u = (uint32_t)i;
        float x;
        memcpy(&x, &u, 4);
        const uint32_t t = u & 0x7fffffffu;
        const bool normal = tge::half_is_normal(x);
        r += normal != (t >= 0x38800000u && t < 0x47800000u);
        if (!normal) continue;
        ++a;
        w += tge::normal_to_half(x) != tge::float_to_half_ref(x);
      }
      accepted[k] = a;
      wrong[k] = w;
      range[k] = r;
    });
  unsigned long long a = 0, w = 0, r = 0;
  for (unsigned k = 0; k < n; ++k) {
    threads[k].join();
    a += accepted[k];
    w += wrong[k];
    r += range[k];
  }
  printf("{\"accepted\": %llu, \"mismatches\": %llu, \"range_errors\": %llu}\n", a, w, r);
  return w || r ? 1 : 0;
}
