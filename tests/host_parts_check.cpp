// Host check of how HostPool cuts a range: no more parts than threads (callers keep
// one record per part), part indices below width(), every byte in exactly one
// part; at lengths around multiples of the threads' 4 KiB pieces above all.
// Prints "OK" or the first mismatch.
#include <atomic>
#include <cstdio>
#include <vector>

#include "../ngap_amd/csrc/host_pool.h"

using ngapamd::HostPool;

int main() {
  for (unsigned helpers = 0; helpers <= 7; helpers++) {
    HostPool pool(helpers);
    const size_t w = pool.width();
    std::vector<size_t> lens = {1, 4095, 4096, 4097, (256u << 10) - 1, 256u << 10, (512u << 10) + 1};
    for (size_t k : {64u, 65u, 128u, 255u})      // pieces of 4 KiB per part
      for (size_t parts = 1; parts <= 8; parts++)
        for (int d : {-1, 0, 1, 7, 4095, 4097}) lens.push_back(parts * k * 4096 + d);
    for (size_t n : lens) {
      const size_t step = pool.part_bytes(n), parts = (n + step - 1) / step;
      if (parts > w) {
        std::printf("%zu bytes: %zu parts for %zu threads\n", n, parts, w);
        return 1;
      }
      std::atomic<size_t> bytes{0}, most{0};
      pool.run_parts(n, [&](size_t i, size_t a, size_t b) {
        bytes += b - a;
        for (size_t m = most; i > m && !most.compare_exchange_weak(m, i);) {}
      });
      if (bytes != n || most >= w) {
        std::printf("%zu bytes: %zu covered, part %zu of %zu\n", n, (size_t)bytes, (size_t)most, w);
        return 1;
      }
    }
  }
  std::printf("OK\n");
  return 0;
}
