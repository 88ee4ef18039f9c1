// Device-side structures shared by the HIP kernels and the host runtime.
#pragma once

#include <cstdint>

#include "layout.h"

#if defined(__HIPCC__)
#define NGAP_HD __host__ __device__
#else
#define NGAP_HD
#endif

namespace ngapamd {

struct DevImage {
  const GroupMeta *meta;
  const int32_t *succ4;      // kRecWords per record (ids, then tests; two int4 loads)
  const uint32_t *cls;       // 8 per state
  const int32_t *sod;
  const uint32_t *beg[kMaxMemoDepth];
  const uint32_t *nrep[kMaxMemoDepth];
  const int32_t *list[kMaxMemoDepth];
  const uint32_t *filt[kMaxMemoDepth];  // next-byte filter of each list entry
  const uint32_t *sel[kMaxMemoDepth];  // rank tables of depths 2 and 3
  const uint32_t *mask1;     // 16 words per group (layout.h)
  // cross-group root index (layout.h)
  const uint32_t *xr1, *xe1, *xmask1, *xr2, *xe2, *xsod, *xs3, *xp3, *xf3, *xb3, *x2rep;
  uint32_t n_xsod;
};

// One batched work item: roots at positions [begin, end) of the chunk
// [cstart, cend) scanned by group `group`; descendants run to cend.  Bit 0 of
// flags seeds the group's start-of-data states at cstart.
struct Task {
  uint32_t group, cstart, cend, begin, end, flags;
};
constexpr uint32_t kTaskSeedStart = 1;
// Work-item overflow flags: the worklist spill area filled up (the item's
// results are incomplete: fallback or error), or its root-pass area did (it
// is re-run without a root pass).
constexpr uint32_t kSpillOverflow = 1, kRootOverflow = 2;
// Task.group of a work item that scans its window for every group at once
// (roots from the cross-group index, memo depth >= 2).
constexpr uint32_t kAllGroups = 0xFFFFFFFFu;

// A piece of a work item for the root pass (k_roots): roots at positions
// [begin, end) of work item `task`; flags as Task.flags (the first piece of a
// work item carries its start-of-data seeding).
struct RootPiece {
  uint32_t task, begin, end, flags;
};

struct KParams {
  DevImage img;
  const uint8_t *input;
  uint32_t chunk_len, num_seg, num_groups;
  // divisibility by chunk_len (> 0): its odd part's inverse modulo 2^32, its
  // power of two, and floor((2^32 - 1) / chunk_len)
  uint32_t div_inverse, div_shift, div_most;
  // Request runs (chunk_len 0): bit p set when position p is the last of its
  // request, so an item of any request finds its chunk end (nullable: then a
  // wave's current work item gives it)
  const uint32_t *last_map;
  int32_t memo_depth;      // 1..3, d-gram roots
  int32_t is_dup;
  int32_t dedup;
  int32_t priv_limit;      // in-lane continuation steps, -1 = unlimited
  int32_t active_threshold;  // continue in-lane only while more lanes than
                             // this are busy (--active-threshold)
  int32_t report_off;
  uint32_t ring_cap;       // LDS ring entries per wave (power of two)
  uint32_t root_batch;     // positions whose roots one step takes (per-group
                           // roots; 1 = NAPgroups' one position at a time)
  unsigned long long *report_count;
  uint64_t *reports;
  uint64_t report_cap;
  uint64_t *spill;
  uint32_t spill_cap;      // items per wave
  uint32_t *overflow;      // plain: per unit; batched: per task
  uint32_t *overflow_count;  // units / tasks that set their overflow flag
  unsigned long long *items;   // expanded items (statistic): kItemLanes lanes
  const Task *tasks;        // nullable: work items generated from their index
  // Generated work items (tasks == nullptr): chunks cut into windows of
  // gen_window positions; all-group work items (gen_cross) ordered by
  // (chunk, window), else one group per work item ordered by (chunk, group,
  // window).
  uint32_t gen_window;
  int32_t gen_cross;
  const uint32_t *task_order;  // nullable
  uint32_t num_tasks;
  int32_t even;            // the work items cost about the same (all-group windows)
  uint32_t *task_head;     // kQueues claim counters, kQueueStride words apart
  unsigned long long *task_items;  // nullable, per task
  uint32_t waves_per_block;
  // k_scan: every work item is an all-group one (scan), and the last input
  // position an 8-byte load may start at
  int32_t scan;
  uint32_t load_last;
  // Root pass (nullable root_items = off): k_roots writes the root items of
  // work item t to root_items[root_off[t] .. root_off[t + 1]), counting them
  // in root_count[t]; the streaming kernel then expands them instead of
  // computing roots.
  const RootPiece *pieces;
  uint32_t num_pieces;
  const uint64_t *root_off;
  uint64_t *root_items;
  unsigned long long *root_count;
};

inline void set_chunk_len(KParams &P, uint32_t len) {
  P.chunk_len = len;
  P.div_shift = (uint32_t)__builtin_ctz(len);
  const uint32_t odd = len >> P.div_shift;
  uint32_t x = odd;  // Newton: correct to 3 bits, doubled each time
  for (int i = 0; i < 4; i++) x *= 2 - odd * x;
  P.div_inverse = x;
  P.div_most = 0xFFFFFFFFu / len;
}

constexpr uint32_t kWave = 64;
constexpr uint32_t kMaxOpen = 8;  // work items a wave overlaps (k_batched)
// LDS entries per wave: report buffer, de-duplication cache (power of two)
constexpr uint32_t kRbuf = 128, kDc = 256;
// The work items that are no workgroup's own are split by XCD: workgroup b runs
// on XCD b % 8, and queue q holds every eighth of them; each claim counter has
// its own 128-byte line.
constexpr uint32_t kQueues = 8, kQueueStride = 32;
// Work items in rows: row `row` of the workgroups' own items has one for each of
// `wgs` workgroups, a row of the queues' one for each queue.  Each row starts one
// column further, so that work items whose cost has a period (groups in a fixed
// order, an input in records: of eight above all) are not all one workgroup's or
// one XCD's.  With column = workgroup in every row, work items heavy eight apart
// took 0.190 ms (a long automaton and seven short, 8,192 windows of 4 KiB, depth 2)
// and 0.048 (8 MiB in windows of 1,024 bytes, every eighth dense), and take 0.150
// and 0.029; alike ones are unchanged.
NGAP_HD inline uint64_t own_item(uint32_t row, uint32_t workgroup, uint32_t wgs) {
  uint32_t col = workgroup + (wgs >= kQueues ? row % kQueues : 0u);
  if (col >= wgs) col -= wgs;
  return (uint64_t)row * wgs + col;
}
NGAP_HD inline uint64_t queue_item(uint32_t row, uint32_t queue, uint32_t queues) {
  const uint32_t col = queues == kQueues ? (queue + row) % kQueues : queue;
  return (uint64_t)row * queues + col;
}
constexpr uint32_t kBlockThreads = 256;
constexpr uint32_t kPlainWaves = 16;  // of a unit in k_plain, at most
// Counters of a run (one buffer per run context, cleared by k_reset): bytes
// 0-31 hold the report count and the count of overflowed work items (word
// 3), byte 128 on the queue claim counters, then kItemLanes lines of
// expanded-item counts, one 64-bit word at the start of each line:
// the waves of workgroup b add theirs at lane b % kItemLanes and the host
// sums the lanes.  A single count that every wave adds to as it ends costs
// 5-8 % of a launch of the streaming kernel: atomics on one address
// serialise.
constexpr uint32_t kItemLanes = 32, kItemStride = 16;  // stride in 64-bit words
constexpr uint32_t kItemsWord = (128 + kQueues * kQueueStride * 4) / 8;
constexpr uint32_t kCounterBytes = (kItemsWord + kItemLanes * kItemStride) * 8;
NGAP_HD inline unsigned long long items_sum(const unsigned long long *counters) {
  unsigned long long n = 0;
  for (uint32_t k = 0; k < kItemLanes; k++) n += counters[kItemsWord + k * kItemStride];
  return n;
}

// Work item t of a generated schedule (KParams::gen_window).
NGAP_HD inline Task gen_task(const KParams &P, uint32_t t) {
  const uint32_t L = P.chunk_len, win = P.gen_window;
  const uint32_t per_chunk = (L + win - 1) / win;
  const uint32_t per_unit = P.gen_cross ? per_chunk : per_chunk * P.num_groups;
  const uint32_t c = t / per_unit, r = t % per_unit;
  const uint32_t g = P.gen_cross ? kAllGroups : r / per_chunk, w = r % per_chunk;
  Task T;
  T.group = g;
  T.cstart = c * L;
  T.cend = T.cstart + L;
  T.begin = T.cstart + w * win;
  T.end = T.begin + win < T.cend ? T.begin + win : T.cend;
  T.flags = (w == 0 && (c == 0 || P.is_dup)) ? kTaskSeedStart : 0u;
  return T;
}

// Batched kernel a launch of P runs: 0 k_batched (one open work item per
// wave: per-work-item traces, or request runs without a last-byte map), 1
// k_batched_stream of engine runs, 2 k_expand (after the root pass), 3
// k_batched_stream of request runs (last-byte map), 4 k_batched_stream of
// generated work items, 5 and 6 k_scan (KParams::scan) of engine runs and of
// generated work items.
constexpr int kBatchedKinds = 7;
NGAP_HD inline int batched_kind(const KParams &P) {
  if (P.task_items || (!P.chunk_len && !P.last_map)) return 0;
  if (P.root_items) return 2;
  if (!P.chunk_len) return 3;
  if (P.scan) return P.tasks ? 5 : 6;
  return P.tasks ? 1 : 4;
}

// LDS bytes per wave: what has a fixed size first (so that it lies at constant
// offsets from one base), then the ring.  Report buffer and de-duplication
// cache, then: list positions in work (65 + 3 x 64 words), the root masks and
// the open work items;
constexpr uint32_t kWaveFixed = (kRbuf + kDc) * 8 + (65 + 3 * kWave + 16 + kMaxOpen + 1) / 2 * 8;
NGAP_HD constexpr uint32_t wave_lds_bytes(uint32_t ring) { return kWaveFixed + ring * 8; }

// in k_scan: 64 marks, the waiting 3-grams (a wave's width less one and a search
// of 128 positions more) and the open work items;
// the groups' bases lie before all waves.  With 1,024 groups four workgroups
// fit a CU's 160 KiB.
constexpr uint32_t kKeyCap = 3 * kWave;
constexpr uint32_t kScanFixed = (kRbuf + kDc) * 8 + kWave * 4 + kKeyCap * 8 + kMaxOpen * 4;
NGAP_HD constexpr uint32_t scan_table_bytes(uint32_t groups) { return (groups * 8 + 15) / 16 * 16; }
NGAP_HD constexpr uint32_t scan_wave_bytes(uint32_t ring) { return kScanFixed + ring * 8; }

constexpr uint32_t kMaxGroups = 1024;  // ten group bits in a report id
// LDS ring entries per wave: by default, and the range of ring_capacity
constexpr uint32_t kRing = 256, kMinRing = 64, kMaxRing = 2048;
// LDS bytes of a launch of the batched kernel `kind` over `groups` groups, and of
// the other kernels with `waves` waves a workgroup; every size is within
// kMaxLds, which each kernel's limit is set to (set_lds_limit).
constexpr uint32_t lds_bytes(uint32_t ring = kRing, uint32_t waves = kBlockThreads / kWave) {
  return 16 + waves * wave_lds_bytes(ring);
}
constexpr uint32_t batched_lds(uint32_t ring, int kind, uint32_t groups) {
  return kind < 5 ? lds_bytes(ring)
                  : 16 + scan_table_bytes(groups) + kBlockThreads / kWave * scan_wave_bytes(ring);
}
constexpr uint32_t larger(uint32_t a, uint32_t b) { return a > b ? a : b; }
constexpr uint32_t kMaxLds = larger(larger(lds_bytes(kMaxRing), lds_bytes(kRing, kPlainWaves)),
                                    batched_lds(kMaxRing, 5, kMaxGroups));
static_assert(kMaxLds <= 160 * 1024, "a workgroup's LDS");

}  // namespace ngapamd
