// Host check of what the launches are sized by (ngap_amd/csrc/kernels.h): the
// dynamic LDS of every kernel's launches is within the limit set for it and the
// device's; the rows of work items are permutations (each item is claimed once,
// the last, incomplete row ends every queue) and spread periodic costs.  Prints
// "OK" or what is wrong.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../ngap_amd/csrc/kernels.h"

using namespace ngapamd;

static int fails = 0;

static void lds(const char *what, uint32_t bytes) {
  if (bytes <= kMaxLds && bytes <= 160 * 1024) return;
  std::printf("%s: %u bytes of LDS, limit %u\n", what, bytes, kMaxLds);
  fails++;
}

// Claims of n work items by `wgs` workgroups, `per` own rows, as the kernels make
// them: own items while their row has them, then the queue's until one is missing.
static void claims(uint64_t n, uint32_t wgs, uint32_t per) {
  const uint32_t queues = std::min(kQueues, wgs);
  std::vector<int> seen(n, 0);
  for (uint32_t b = 0; b < wgs; b++)
    for (uint32_t i = 0; i < per; i++) {
      const uint64_t t = own_item(i, b, wgs);
      if (t >= n) break;
      seen[t]++;
    }
  for (uint32_t q = 0; q < queues; q++)
    if ((uint64_t)per * wgs + q < n)
      for (uint32_t i = 0;; i++) {
        const uint64_t t = (uint64_t)per * wgs + queue_item(i, q, queues);
        if (t >= n) break;
        seen[t]++;
      }
  for (uint64_t t = 0; t < n; t++)
    if (seen[t] != 1) {
      std::printf("%llu items, %u workgroups, %u rows: item %llu claimed %d times\n",
                  (unsigned long long)n, wgs, per, (unsigned long long)t, seen[t]);
      fails++;
      return;
    }
}

// Of work items heavy `period` apart: no workgroup and no queue has more than
// twice its share, and one.
static void spread(uint32_t wgs, uint32_t rows, uint32_t period) {
  for (uint32_t b = 0; b < wgs; b++) {
    uint32_t heavy = 0;
    for (uint32_t i = 0; i < rows; i++) heavy += own_item(i, b, wgs) % period == 0;
    if (heavy > 2 * rows / period + 1) {
      std::printf("period %u: workgroup %u of %u has %u of %u heavy\n", period, b, wgs, heavy, rows);
      fails++;
      return;
    }
  }
  for (uint32_t q = 0; q < kQueues; q++) {
    uint32_t heavy = 0;
    for (uint32_t i = 0; i < 1000; i++) heavy += queue_item(i, q, kQueues) % period == 0;
    if (heavy > 2 * 1000 / period + 1) {
      std::printf("period %u: queue %u has %u of 1000 heavy\n", period, q, heavy);
      fails++;
      return;
    }
  }
}

int main() {
  for (uint32_t wgs : {1u, 2u, 3u, 7u, 8u, 9u, 12u, 16u, 63u, 64u, 100u, 1280u})
    for (uint32_t per : {0u, 1u, 4u, 6u, 9u, 20u})
      for (uint64_t n : {(uint64_t)0, (uint64_t)1, (uint64_t)per * wgs, (uint64_t)per * wgs + 1,
                         (uint64_t)per * wgs + 7, (uint64_t)per * wgs + 8,
                         (uint64_t)per * wgs + 9, (uint64_t)per * wgs + 1001})
        claims(n, wgs, per);
  // fewer items than the own rows: every row is started, the last is incomplete
  for (uint32_t wgs : {1u, 5u, 8u, 13u, 64u})
    for (uint64_t n = 1; n < 400; n++) claims(n, wgs, (uint32_t)((n + wgs - 1) / wgs));
  for (uint32_t wgs : {8u, 64u, 1024u, 1280u})
    for (uint32_t rows : {4u, 6u, 24u, 100u})
      for (uint32_t period : {2u, 4u, 8u}) spread(wgs, rows, period);
  for (uint32_t waves = kBlockThreads / kWave; waves <= kPlainWaves; waves *= 2)
    lds("plain", lds_bytes(kRing, waves));
  for (uint32_t ring = kMinRing; ring <= kMaxRing; ring *= 2)
    for (int kind = 0; kind < kBatchedKinds; kind++)
      for (uint32_t groups = 1; groups <= 1024; groups++) lds("batched", batched_lds(ring, kind, groups));
  if (!fails) std::printf("OK\n");
  return fails != 0;
}
