// Host check of what the launches are sized by (ngap_amd/csrc/kernels.h): the
// dynamic LDS of every kernel's launches is within the limit set for it and the
// device's.  Prints "OK" or what is wrong.
#include <cstdio>

#include "../ngap_amd/csrc/kernels.h"

using namespace ngapamd;

static int fails = 0;

static void lds(const char *what, uint32_t bytes) {
  if (bytes <= kMaxLds && bytes <= 160 * 1024) return;
  std::printf("%s: %u bytes of LDS, limit %u\n", what, bytes, kMaxLds);
  fails++;
}

int main() {
  for (uint32_t waves = kBlockThreads / kWave; waves <= kPlainWaves; waves *= 2)
    lds("plain", lds_bytes(kRing, waves));
  for (uint32_t ring = kMinRing; ring <= kMaxRing; ring *= 2)
    for (int kind = 0; kind < kBatchedKinds; kind++)
      for (uint32_t groups = 1; groups <= 1024; groups++) lds("batched", batched_lds(ring, kind, groups));
  if (!fails) std::printf("OK\n");
  return fails != 0;
}
