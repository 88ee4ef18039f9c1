// HIP kernels for gfx950 (wave64): the non-blocking (state, offset) worklist
// engine.
//
// Reference behaviour (what is computed): the worklist kernels
// advanceAndFilterNonBlocking{NAP,,R1,R2,Prec,All}Groups
// (code/src/ngap/kernel_bap.cu:10-185, kernel_ngap_O1.cu:10-185,
// kernel_ngap_O4.cu:9-548, kernel_ngap_O3.cu:10-295, kernel_ngap_OA.cu:10-374):
// an item (v, p) means state v matched input[p]; expanding it tests every
// successor u of v against input[p+1], reports u when it reports, and enables
// (u, p+1).  All-input states are enabled at every position; start-of-data
// states at the first position of chunk 0 (or of every chunk when the input
// was duplicated).  The report set is the reference's; item order is free.
//
// How it is computed here (MI355X-first, not the reference's structure):
//  * Each wave owns a ring of items in LDS.  Pushes are compacted with
//    ballot + mbcnt (one ring slot computation per wave, no atomics at all:
//    head/tail are wave-uniform registers).  Items beyond the ring go to a
//    per-wave HBM spill area and come back when the ring runs low.
//  * Idle lanes refill from the ring every step, so a wave stays converged
//    and busy without block barriers.
//  * A lane keeps the first surviving successor of its item in registers and
//    continues with it (work privatization generalised to whole chains; the
//    reference expands one more level, kernel_ngap_OA.cu:96-138).
//  * Roots come from the memo tables: one lookup per position gives the
//    states matched d-1 positions later (prefix memoization,
//    kernel_ngap_OA.cu:243-310), flattened across the wave with a prefix sum.
//  * Reports are compacted into a per-wave LDS buffer and flushed with one
//    global atomic per flush (the reference: one atomic per report,
//    kernel_helper.h:78-104).
//  * (state, offset) items of states with two or more incoming edges pass a
//    lossy LDS cache (64-bit atomic exchange): an exact duplicate seen
//    recently is dropped.  A duplicate is never needed (set semantics), and a
//    first occurrence is never dropped.
//  * The batched engine is a persistent grid whose waves pull work items
//    (a window of one chunk, for one group or for all groups) from eight
//    XCD-local queues; an all-group work item takes the roots of every group
//    from the cross-group 2-/3-gram index, one lookup per position.
//  * The loads of a step (input bytes, index offsets, a record and its class
//    words) are issued unconditionally at valid stand-in addresses and
//    selected afterwards, so they go out together: the engine is bound by the
//    latency of dependent gathers.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace ngapamd {

#define NGAP_DEV __device__ __forceinline__
// Branch weights: what a wave seldom does goes out of line.  A taken branch
// costs a lone wave as much as a dozen instructions (the fetch starts over), so
// the common path falls through.
#define NGAP_SELDOM(x) __builtin_expect((x) != 0, 0)
#define NGAP_MOSTLY(x) __builtin_expect((x) != 0, 1)

NGAP_DEV uint32_t lane_id() {
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}
NGAP_DEV uint32_t mask_rank(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
NGAP_DEV uint64_t wballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// A value that every lane is to have from one lane, read into a scalar
// register.  What steers the wave (claims, queue ends, counts) must come this
// way and not from a shuffle: a shuffled value is a vector to the compiler, the
// branches on it are divergent, and every counter that a loop carries through
// them moves to vector registers and vector instructions.
NGAP_DEV uint32_t from_first(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }
NGAP_DEV uint64_t from_first(uint64_t x) {
  return (uint64_t)from_first((uint32_t)x) | ((uint64_t)from_first((uint32_t)(x >> 32)) << 32);
}
NGAP_DEV uint32_t from_last(uint32_t x) { return __builtin_amdgcn_readlane(x, 63); }
NGAP_DEV void wsync() { __builtin_amdgcn_wave_barrier(); }

NGAP_DEV uint32_t wave_incl_scan(uint32_t x, uint32_t lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t y = __shfl_up(x, off, 64);
    if (lane >= (uint32_t)off) x += y;
  }
  return x;
}

// Inclusive scans over the wave on the DPP network: shifts inside rows of 16
// lanes, then the last lane of a row broadcast to the rows after it.
template <int Ctrl, int Rows>
NGAP_DEV uint32_t dpp(uint32_t x) {  // 0 where the source lane does not exist
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, Ctrl, Rows, 0xF, false);
}
template <class Op>
NGAP_DEV uint32_t dpp_scan(uint32_t x, Op op) {  // op(x, 0) = x
  x = op(x, dpp<0x111, 0xF>(x));
  x = op(x, dpp<0x112, 0xF>(x));
  x = op(x, dpp<0x114, 0xF>(x));
  x = op(x, dpp<0x118, 0xF>(x));
  x = op(x, dpp<0x142, 0xA>(x));
  return op(x, dpp<0x143, 0xC>(x));
}

// The kernel's parameters read again from memory, for the paths that a wave
// seldom takes: what only they need does not occupy scalar registers in
// between.  (Every kernel's only argument is KParams.)
NGAP_DEV const KParams &cold_params() {
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const KParams *)p;
}

// A wave's expanded items, added at its workgroup's lane of the count.
NGAP_DEV void add_items(unsigned long long n) {
  const KParams &P = cold_params();
  atomicAdd(P.items + (blockIdx.x % kItemLanes) * kItemStride, n);
}

struct WaveState {
  uint64_t *ring;
  uint64_t *rbuf;
  uint64_t *dc;
  uint32_t *sh_pref;  // 65
  uint32_t *sh_beg;   // 64
  uint32_t *sh_pos;   // 64
  uint32_t *sh_tag;   // 64
  uint32_t *mask1;    // 16: root bytes, then reporting depth-1 bytes (layout.h)
  uint32_t *open;     // kMaxOpen: work items whose items may still be queued
  uint32_t n_open;
  uint32_t head, tail, rn, spill_n;
  uint32_t lane, wave;
  bool overflow;
  unsigned long long items;
  // root pass: the work item's area of root_items and its item count
  uint64_t *out;
  unsigned long long *out_count;
  uint64_t out_cap;
  // current (group, chunk)
  uint32_t g, gtag, rec_base, cls_base, cstart, cend;
};

NGAP_DEV bool class_has(const KParams &P, uint32_t cls_base, uint32_t u, uint32_t b) {
  return (P.img.cls[(size_t)(cls_base + u) * 8 + (b >> 5)] >> (b & 31)) & 1u;
}

// An item (and a report) is (offset << 32) | (group << 22) | state.
NGAP_DEV uint64_t item_of(uint32_t tagged, uint32_t pos) {
  return ((uint64_t)pos << 32) | tagged;
}

// A 32-byte successor record: four tagged successor ids and their tests.
struct Rec {
  int4 ids;
  uint4 tests;
};

NGAP_DEV Rec load_rec(const KParams &P, uint32_t r) {
  const int4 *R = reinterpret_cast<const int4 *>(P.img.succ4) + (size_t)r * 2;
  Rec x;
  x.ids = R[0];
  const int4 t = R[1];
  x.tests = make_uint4((uint32_t)t.x, (uint32_t)t.y, (uint32_t)t.z, (uint32_t)t.w);
  return x;
}

NGAP_DEV Rec empty_rec() {
  Rec x;
  x.ids = make_int4(-1, -1, -1, -1);
  x.tests = make_uint4(0, 0, 0, 0);
  return x;
}

// Class word a successor test needs (0 when the test word decides alone).
NGAP_DEV uint32_t test_word(const KParams &P, uint32_t cls_base, bool live, int32_t e,
                            uint32_t t, uint32_t b) {
  if (!live || e < 0 || (t & (kTestLiteral | kTestAll))) return 0u;
  return P.img.cls[(size_t)(cls_base + ((uint32_t)e & (uint32_t)kIdMask)) * 8 + (b >> 5)];
}

NGAP_DEV bool test_hit(bool live, int32_t e, uint32_t t, uint32_t word, uint32_t b) {
  if (!live || e < 0) return false;
  if (t & kTestLiteral) return (t & 255u) == b;
  if (t & kTestAll) return true;
  return (word >> (b & 31)) & 1u;
}

// Root pass: the wave's ring is a staging buffer (filled from 0), appended
// to the work item's area of root_items when it fills and at the end of a
// piece.  Items beyond the area's capacity are dropped and the work item is
// marked for the fallback.
NGAP_DEV void flush_stage(const KParams &P, WaveState &W) {
  if (W.tail == 0) return;
  wsync();
  uint64_t base = 0;
  if (W.lane == 0) base = atomicAdd(W.out_count, (unsigned long long)W.tail);
  base = from_first(base);
  for (uint32_t i = W.lane; i < W.tail; i += kWave)
    if (base + i < W.out_cap) W.out[base + i] = W.ring[i];
  if (base + W.tail > W.out_cap) W.overflow = true;
  W.tail = 0;
  wsync();
}

// The wave's spill area and its capacity.
NGAP_DEV uint64_t *spill_area(const WaveState &W, uint32_t &cap) {
  const KParams &P = cold_params();
  cap = P.spill_cap;
  return P.spill + ((size_t)blockIdx.x * P.waves_per_block + W.wave) * cap;
}

template <bool Stage = false>
NGAP_DEV void push(const KParams &P, WaveState &W, bool pred, uint64_t item) {
  uint64_t m = wballot(pred);
  if (m == 0) return;
  uint32_t cnt = __popcll(m);
  uint32_t r = mask_rank(m);
  if (Stage) {
    if (W.tail + cnt > P.ring_cap) flush_stage(P, W);
    if (pred) W.ring[W.tail + r] = item;
    W.tail += cnt;
    wsync();
    return;
  }
  // the barriers inside the branches keep the compiler from folding a lane's
  // condition into the wave's, which would make the counters vectors
  if (NGAP_MOSTLY(W.tail - W.head + cnt <= P.ring_cap)) {
    if (pred) W.ring[(W.tail + r) & (P.ring_cap - 1)] = item;
    wsync();
    W.tail += cnt;
  } else {
    uint32_t cap;
    uint64_t *spill = spill_area(W, cap);
    if (W.spill_n + cnt <= cap) {
      if (pred) spill[W.spill_n + r] = item;
      wsync();
      W.spill_n += cnt;
    } else {
      W.overflow = true;
    }
  }
  wsync();
}

NGAP_DEV void flush_reports(WaveState &W) {
  if (W.rn == 0) return;
  const KParams &P = cold_params();
  wsync();
  uint64_t base = 0;
  if (W.lane == 0) base = atomicAdd(P.report_count, (unsigned long long)W.rn);
  base = from_first(base);
  if (!P.report_off) {
    for (uint32_t i = W.lane; i < W.rn; i += kWave) {
      const uint64_t idx = base + i;
      if (idx < P.report_cap) P.reports[idx] = W.rbuf[i];
    }
  }
  W.rn = 0;
  wsync();
}

// Report encoding on the device: (offset << 32) | (state | group << 22), so a
// plain numeric sort gives the reference's (offset, id) order.
NGAP_DEV void emit(const KParams &P, WaveState &W, bool pred, uint64_t val) {
  uint64_t m = wballot(pred);
  if (m == 0) return;
  uint32_t cnt = __popcll(m);
  if (NGAP_SELDOM(W.rn + cnt > kRbuf)) flush_reports(W);
  if (pred) W.rbuf[W.rn + mask_rank(m)] = val;
  W.rn += cnt;
  wsync();
}

// Queues an item unless its next byte shows that it expands to nothing (its
// state's next-byte filter, layout.h); such an item is counted as expanded,
// which is all that expanding it would have done.
template <bool Stage = false>
NGAP_DEV void push_filtered(const KParams &P, WaveState &W, bool keep, uint32_t filt,
                            uint32_t next, uint64_t item) {
  const bool pass = keep & (((filt >> filter_bit(next)) & 1u) != 0);
  W.items += __popcll(wballot(keep & !pass));
  push<Stage>(P, W, pass, item);
}

NGAP_DEV uint32_t min_u(uint32_t a, uint32_t b) { return a < b ? a : b; }

NGAP_DEV bool dedup_fresh(const KParams &P, WaveState &W, uint64_t key) {
  uint32_t h = (uint32_t)((key * 0x9E3779B97F4A7C15ull) >> 40) & (kDc - 1);
  unsigned long long old = atomicExch((unsigned long long *)&W.dc[h], (unsigned long long)key);
  return old != key;
}

// Spilled items return to the ring when it runs low.
NGAP_DEV void refill_from_spill(const KParams &P, WaveState &W) {
  uint32_t room = P.ring_cap - (W.tail - W.head);
  uint32_t k = W.spill_n < room ? W.spill_n : room;
  uint32_t from = W.spill_n - k, cap;
  const uint64_t *spill = spill_area(W, cap);
  for (uint32_t i = W.lane; i < k; i += kWave)
    W.ring[(W.tail + i) & (P.ring_cap - 1)] = spill[from + i];
  W.tail += k;
  W.spill_n = from;
  wsync();
}

// Processes a variable number of memo-list entries per lane as one flat index
// space (prefix sum over the wave), 64 entries per step.  Every entry that
// reports is emitted; entries are also pushed as items unless the lane's
// list is report-only (bit 31 of beg), the state has no successors, or the
// position is the chunk's last, or (Filter) its next byte cannot match.
template <bool Stage = false, bool Filter = true>
NGAP_DEV void flatten(const KParams &P, WaveState &W, uint32_t cnt, uint32_t beg,
                      uint32_t pos, uint32_t gtag, const int32_t *list,
                      const uint32_t *filt) {
  const uint32_t last = W.cend - 1;
  if (wballot(cnt > 1u) == 0) {
    // at most one entry per lane (the common case): no prefix sum
    const bool ok = cnt == 1u;
    if (wballot(ok) == 0) return;
    const int32_t e = ok ? list[beg & 0x7fffffffu] : 0;
    uint32_t f = 0, next = 0;
    if (Filter) {
      f = ok ? filt[beg & 0x7fffffffu] : 0;
      next = P.input[ok ? min_u(pos + 1, last) : last];
    }
    const uint64_t it = item_of(((uint32_t)e & (uint32_t)kIdMask) | gtag, pos);
    emit(P, W, ok && (e & kFlagReport), it);
    bool keep = ok && !(beg >> 31) && !(e & kFlagDeadEnd) && (pos + 1 < W.cend);
    if (keep && P.dedup && (e & kFlagDedup)) keep = dedup_fresh(P, W, it);
    if (Filter) push_filtered<Stage>(P, W, keep, f, next, it);
    else push<Stage>(P, W, keep, it);
    return;
  }
  uint32_t incl = wave_incl_scan(cnt, W.lane);
  uint32_t total = from_last(incl);
  if (total == 0) return;
  W.sh_pref[W.lane] = incl - cnt;
  W.sh_beg[W.lane] = beg;
  W.sh_pos[W.lane] = pos;
  W.sh_tag[W.lane] = gtag;
  if (W.lane == 63) W.sh_pref[64] = total;
  wsync();
  for (uint32_t base = 0; base < total; base += kWave) {
    uint32_t j = base + W.lane;
    bool ok = j < total;
    int32_t e = 0;
    uint32_t ppos = 0, tg = 0, f = 0, next = 0;
    bool ronly = true;
    if (ok) {
      int lo = 0, hi = 64;  // largest o with pref[o] <= j (pref[64] = total > j)
      while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (W.sh_pref[mid] <= j) lo = mid;
        else hi = mid - 1;
      }
      const uint32_t bg = W.sh_beg[lo];
      ronly = bg >> 31;
      const uint32_t at = (bg & 0x7fffffffu) + (j - W.sh_pref[lo]);
      e = list[at];
      ppos = W.sh_pos[lo];
      if (Filter) {
        f = filt[at];
        next = P.input[min_u(ppos + 1, last)];
      }
      tg = W.sh_tag[lo];
    }
    const uint32_t u = ((uint32_t)e & (uint32_t)kIdMask) | tg;
    emit(P, W, ok && (e & kFlagReport), item_of(u, ppos));
    bool keep = ok && !ronly && !(e & kFlagDeadEnd) && (ppos + 1 < W.cend);
    if (keep && P.dedup && (e & kFlagDedup)) keep = dedup_fresh(P, W, item_of(u, ppos));
    if (Filter) push_filtered<Stage>(P, W, keep, f, next, item_of(u, ppos));
    else push<Stage>(P, W, keep, item_of(u, ppos));
  }
  wsync();
}

// Roots for positions [p0, pend): one lane per position.  A position whose
// byte starts no root costs one load and one bit test.  A lane uses the
// deepest memo level that fits before the chunk end (kernel_ngap_OA.cu:243-
// 244); shallower levels contribute their reports only.  With depth >= 2 the
// independent loads of all levels are issued together (input bytes, then the
// rank pairs, then the list ranges) and the depth-1 lists are read only for
// bytes whose list reports.
// Loads in the root and expansion steps are issued unconditionally, at a
// valid address when a lane does not need the value (index 0, or the chunk's
// last byte), and the value is selected afterwards: the loads of a step then
// go out together instead of one branch (and one wait) at a time.
// Deep: the lists of depth 2 and 3 with their entries' filters.  Where a unit's
// waves take their positions one batch after the other (drain) they spare a step
// too seldom (1,024 automata of up to 5,000 states, 2 MiB, plain: depth 2 4.91 ms
// without and 5.05 with them, depth 3 4.73 and 4.84).  Work items whose roots and
// expansions overlap (drain_stream) gain 2 % by them, and at depth 1 they always
// pay (11.1 and 8.7 ms plain, 10.9 and 8.1 batched, with 50,000 states).
template <bool Stage = false, bool Deep = true>
NGAP_DEV void roots(const KParams &P, WaveState &W, uint32_t p0, uint32_t pend) {
  const uint8_t *in = P.input;
  const uint32_t p = p0 + W.lane;
  const bool act = p < pend;
  const uint32_t left = act ? W.cend - p : 0u;
  const uint32_t k = left < (uint32_t)P.memo_depth ? left : (uint32_t)P.memo_depth;
  const uint32_t pc = act ? p : p0, last = W.cend - 1;
  const uint32_t b0 = in[pc];
  const uint32_t b1 = in[min_u(pc + 1, last)];
  const uint32_t b2 = in[min_u(pc + 2, last)];
  const bool has = act && ((W.mask1[b0 >> 5] >> (b0 & 31)) & 1u);
  if (wballot(has) == 0) return;
  const uint32_t kReportOnly = 1u << 31;
  if (P.memo_depth < 2) {  // depth 1: all-input states matching b0 become items
    const uint32_t li = W.g * 256u + b0;
    const uint32_t beg = P.img.beg[0][li], end = P.img.beg[0][li + 1];
    flatten<Stage>(P, W, has ? end - beg : 0u, beg, p, W.gtag, P.img.list[0], P.img.filt[0]);
    return;
  }
  // rank pair of the 2-gram (and the depth-1 reports of rare bytes)
  const uint32_t key = (b0 << 8) | b1;
  const uint2 w2 = reinterpret_cast<const uint2 *>(P.img.sel[1])[(size_t)W.g * 2048 + (key >> 5)];
  const uint32_t bit2 = key & 31;
  const int32_t li2 = has && k >= 2 && ((w2.x >> bit2) & 1u)
                          ? (int32_t)(w2.y + __popc(w2.x & ((1u << bit2) - 1u)))
                          : -1;
  const bool rep1 = has && ((W.mask1[8 + (b0 >> 5)] >> (b0 & 31)) & 1u);
  if (wballot(rep1)) {  // depth 1: reporting entries only (the last position included)
    uint32_t beg = 0, cnt = 0;
    if (rep1) {
      const uint32_t li = W.g * 256u + b0;
      beg = P.img.beg[0][li] | kReportOnly;
      cnt = P.img.nrep[0][li];
    }
    flatten<Stage>(P, W, cnt, beg, p, W.gtag, P.img.list[0], P.img.filt[0]);
  }
  const bool has2 = li2 >= 0;
  if (wballot(has2) == 0) return;
  // depth-2 list range and the depth-3 rank pair (some lane has a depth-2
  // list, so index 0 and 1 are valid stand-ins)
  const uint32_t l2 = has2 ? (uint32_t)li2 : 0u;
  const uint32_t beg2r = P.img.beg[1][l2], end2 = P.img.beg[1][l2 + 1];
  const uint32_t nrep2 = P.img.nrep[1][l2];
  int32_t li3 = -1;
  if (P.memo_depth >= 3) {
    const uint2 w3 = reinterpret_cast<const uint2 *>(P.img.sel[2])[(size_t)l2 * 8 + (b2 >> 5)];
    const uint32_t bit3 = b2 & 31;
    li3 = has2 && k >= 3 && ((w3.x >> bit3) & 1u)
              ? (int32_t)(w3.y + __popc(w3.x & ((1u << bit3) - 1u)))
              : -1;
  }
  uint32_t cnt2 = has2 ? (k == 2 ? end2 - beg2r : nrep2) : 0u;
  const uint32_t beg2 = k == 2 ? beg2r : (beg2r | kReportOnly);
  uint32_t beg3 = 0, cnt3 = 0;
  if (wballot(li3 >= 0)) {
    const uint32_t l3 = li3 >= 0 ? (uint32_t)li3 : 0u;
    const uint32_t b3 = P.img.beg[2][l3], e3 = P.img.beg[2][l3 + 1];
    beg3 = b3;
    cnt3 = li3 >= 0 ? e3 - b3 : 0u;
  }
  flatten<Stage, Deep>(P, W, cnt2, beg2, p + 1, W.gtag, P.img.list[1], P.img.filt[1]);
  if (wballot(cnt3 != 0)) 
    flatten<Stage, Deep>(P, W, cnt3, beg3, p + 2, W.gtag, P.img.list[2], P.img.filt[2]);
}

// Distributes per-lane index ranges [e0, e0 + ecnt) over the wave, 64
// entries per round, and calls f(ok, entry index, owner lane) each round (a
// wave-uniform loop; the owner is found by binary search over the inclusive
// prefix sums held in the lanes).
template <class F>
NGAP_DEV void for_entries(const WaveState &W, uint32_t e0, uint32_t ecnt, F &&f) {
  if (wballot(ecnt > 1u) == 0) {  // at most one entry per lane: its own
    f(ecnt == 1u, e0, W.lane);
    return;
  }
  const uint32_t incl = wave_incl_scan(ecnt, W.lane);
  const uint32_t total = from_last(incl);
  for (uint32_t base = 0; base < total; base += kWave) {
    const uint32_t j = base + W.lane;
    const bool ok = j < total;
    uint32_t lo = 0, hi = 63;  // smallest lane o with incl[o] > j
#pragma unroll
    for (int s = 0; s < 6; s++) {
      const uint32_t mid = (lo + hi) >> 1;
      if (__shfl(incl, (int)mid, 64) > j) hi = mid;
      else lo = mid + 1;
    }
    const uint32_t oi = __shfl(incl, (int)lo, 64);
    const uint32_t oc = __shfl(ecnt, (int)lo, 64);
    const uint32_t oe = __shfl(e0, (int)lo, 64);
    f(ok, oe + j - (oi - oc), lo);
  }
}

// for_entries over two ranges per lane, [a0, a0 + ac) then [b0, b0 + bc)
// (the two halves of a 128-position batch): f(ok, entry index, owner lane,
// range 0 or 1).
template <class F>
NGAP_DEV void for_entries2(const WaveState &W, uint32_t a0, uint32_t ac, uint32_t b0,
                           uint32_t bc, F &&f) {
  const uint32_t n = ac + bc;
  const uint32_t incl = wave_incl_scan(n, W.lane);
  const uint32_t total = from_last(incl);
  for (uint32_t base = 0; base < total; base += kWave) {
    const uint32_t j = base + W.lane;
    const bool ok = j < total;
    uint32_t lo = 0, hi = 63;  // smallest lane o with incl[o] > j
#pragma unroll
    for (int s = 0; s < 6; s++) {
      const uint32_t mid = (lo + hi) >> 1;
      if (__shfl(incl, (int)mid, 64) > j) hi = mid;
      else lo = mid + 1;
    }
    const uint32_t off = j - (__shfl(incl, (int)lo, 64) - __shfl(n, (int)lo, 64));
    const uint32_t oac = __shfl(ac, (int)lo, 64);
    // both bases are read by every lane before the select: a shuffle inside
    // a divergent branch reads nothing from lanes outside that branch
    const uint32_t oa0 = __shfl(a0, (int)lo, 64), ob0 = __shfl(b0, (int)lo, 64);
    const bool second = off >= oac;
    f(ok, second ? ob0 + (off - oac) : oa0 + off, lo, second ? 1u : 0u);
  }
}

// Per-lane state of one position in roots_cross.
struct CrossLane {
  uint32_t p, k, b0, b3, e0, ec, t0, tc, r0, rc;
};

// The loads of one position's lookups, in stages shared by both halves of a
// 128-position batch: input bytes, then the index offsets.
NGAP_DEV void cross_lookup(const KParams &P, const WaveState &W, uint32_t p0, uint32_t pend,
                           CrossLane (&L)[2]) {
  const uint8_t *in = P.input;
  const uint32_t last = W.cend - 1;
  uint32_t b1[2], b2[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t p = p0 + h * kWave + W.lane;
    const bool act = p < pend;
    const uint32_t left = act ? W.cend - p : 0u;
    const uint32_t pc = act ? p : p0;
    L[h].p = p;
    L[h].k = left < (uint32_t)P.memo_depth ? left : (uint32_t)P.memo_depth;
    L[h].b0 = in[pc];
    b1[h] = in[min_u(pc + 1, last)];
    b2[h] = in[min_u(pc + 2, last)];
    L[h].b3 = in[min_u(pc + 3, last)];
  }
  // Depth 3: the 3-gram slots first.  A slot flags the 3-grams whose first
  // byte or first two bytes begin reporting lists of depth 1 or 2 in some
  // group; the byte and 2-gram indexes are read only when some lane has such
  // a 3-gram or fewer than three bytes left in its chunk (for every other
  // lane their ranges are empty).
  bool full = P.memo_depth < 3;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    L[h].t0 = L[h].tc = L[h].e0 = L[h].ec = L[h].r0 = L[h].rc = 0;
    if (P.memo_depth >= 3) {
      const uint32_t k = L[h].k;
      const uint32_t key3 = (L[h].b0 << 16) | (b1[h] << 8) | b2[h];
      const uint2 slot = reinterpret_cast<const uint2 *>(P.img.xs3)[key3];
      L[h].t0 = slot.x;
      L[h].tc = k >= 3 ? (slot.y & ~kSlotPrefixReports) : 0u;
      full = full || (k >= 1 && k < 3) || (k >= 3 && (slot.y & kSlotPrefixReports));
    }
  }
  if (wballot(full) == 0) return;
  uint32_t x2w[2], x2a[2], x2b[2], x1a[2], x1b[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t key2 = (L[h].b0 << 8) | b1[h];
    x2a[h] = P.img.xr2[key2];
    x2b[h] = P.img.xr2[key2 + 1];
    x1a[h] = P.img.xr1[L[h].b0];
    x1b[h] = P.img.xr1[L[h].b0 + 1];
    x2w[h] = P.memo_depth >= 3 ? P.img.x2rep[key2 >> 5] : 0u;
  }
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t k = L[h].k, b0 = L[h].b0, key2 = (b0 << 8) | b1[h];
    // depth-2 lists: the deepest level at depth 2; at depth 3 only where two
    // bytes are left or the 2-gram has reporting depth-2 lists
    const bool need2 = k >= 2 && (P.memo_depth == 2 || k == 2 || ((x2w[h] >> (key2 & 31)) & 1u));
    L[h].e0 = x2a[h];
    L[h].ec = need2 ? x2b[h] - x2a[h] : 0u;
    L[h].r0 = x1a[h];
    L[h].rc = k >= 1 && ((W.mask1[8 + (b0 >> 5)] >> (b0 & 31)) & 1u) ? x1b[h] - x1a[h] : 0u;
  }
}

// One entry per lane at most: the entry and its single list item are loaded
// for both halves before either is emitted.
template <bool Stage = false>
NGAP_DEV void emit_one(const KParams &P, WaveState &W, bool ok, int32_t e, uint32_t filt,
                       uint32_t next, uint32_t pos, uint32_t tag) {
  const uint64_t it = item_of(((uint32_t)e & (uint32_t)kIdMask) | tag, pos);
  emit(P, W, ok && (e & kFlagReport), it);
  bool keep = ok && !(e & kFlagDeadEnd) && (pos + 1 < W.cend);
  if (keep && P.dedup && (e & kFlagDedup)) keep = dedup_fresh(P, W, it);
  push_filtered<Stage>(P, W, keep, filt, next, it);
}

// Roots of every group for positions [p0, pend), pend - p0 <= 128 (cross-
// group work items, memo depth >= 2): one lane per position and half; the
// position's byte selects the groups whose all-input states report on it,
// its 2-gram the depth-2 lists and its 3-gram the depth-3 lists of every
// group.  The same lists as roots() visits group by group, so the same items.
template <bool Stage = false>
NGAP_DEV void roots_cross(const KParams &P, WaveState &W, uint32_t p0, uint32_t pend) {
  const uint32_t kReportOnly = 1u << 31;
  CrossLane L[2];
  cross_lookup(P, W, p0, pend, L);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t p = L[h].p;
    // depth 1: reporting entries only (positions that continue use depth >= 2)
    if (wballot(L[h].rc != 0)) {
      for_entries(W, L[h].r0, L[h].rc, [&](bool ok, uint32_t idx, uint32_t o) {
        const uint32_t pos = __shfl(p, (int)o, 64);
        uint32_t beg = 0, cnt = 0, tag = 0;
        if (ok) {
          const uint32_t li = P.img.xe1[idx];
          beg = P.img.beg[0][li] | kReportOnly;
          cnt = P.img.nrep[0][li];
          tag = (li >> 8) << 22;
        }
        flatten<Stage>(P, W, cnt, beg, pos, tag, P.img.list[0], P.img.filt[0]);
      });
    }
    // depth 2: full lists where it is the deepest level, reports otherwise
    if (wballot(L[h].ec != 0)) {
      const uint32_t k = L[h].k;
      for_entries(W, L[h].e0, L[h].ec, [&](bool ok, uint32_t idx, uint32_t o) {
        const uint32_t pos = __shfl(p, (int)o, 64);
        const uint32_t ko = __shfl(k, (int)o, 64);
        uint32_t beg = 0, cnt = 0, tag = 0;
        if (ok) {
          // (list index, begin, end, reporting entries | group << 22)
          const uint4 e = reinterpret_cast<const uint4 *>(P.img.xe2)[idx];
          tag = (e.w >> 22) << 22;
          beg = e.y;
          cnt = ko == 2 || P.memo_depth == 2 ? e.z - e.y : (e.w & (uint32_t)kIdMask);
          if (!(ko == 2 || P.memo_depth == 2)) beg |= kReportOnly;
        }
        flatten<Stage>(P, W, cnt, beg, pos + 1, tag, P.img.list[1], P.img.filt[1]);
      });
    }
  }
  if (P.memo_depth < 3) return;
  // depth 3 from the 3-gram slots: an inline state is emitted at once; the
  // other slots' (tagged state, group) pairs of both halves are spread over
  // the wave together, one 8-byte load per pair
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const bool inl = (L[h].tc & kSlotInline) != 0;
    emit_one<Stage>(P, W, inl, (int32_t)L[h].t0, slot_filter(L[h].t0, L[h].tc), L[h].b3,
                    L[h].p + 2, (L[h].tc & 1023u) << 22);
    if (inl) L[h].tc = 0;
  }
  if (wballot(L[0].tc != 0 || L[1].tc != 0) == 0) return;
  // some lane has pairs, so pair 0 is a valid stand-in address
  const uint32_t b3 = L[0].b3 | (L[1].b3 << 8);
  for_entries2(W, L[0].t0, L[0].tc, L[1].t0, L[1].tc,
               [&](bool ok, uint32_t idx, uint32_t o, uint32_t h) {
                 const uint2 e = reinterpret_cast<const uint2 *>(P.img.xp3)[ok ? idx : 0u];
                 const uint32_t f = P.img.xf3[ok ? idx : 0u];
                 const uint32_t next = (__shfl(b3, (int)o, 64) >> (8 * h)) & 255u;
                 emit_one<Stage>(P, W, ok, (int32_t)e.x, f, next, p0 + h * kWave + o + 2,
                                 e.y << 22);
               });
}

template <bool Stage = false>
NGAP_DEV void seed_start_of_data(const KParams &P, WaveState &W, uint32_t sod_begin,
                                 uint32_t sod_end) {
  uint32_t b = P.input[W.cstart];
  for (uint32_t i = sod_begin; i < sod_end; i += kWave) {
    uint32_t idx = i + W.lane;
    bool ok = idx < sod_end;
    int32_t e = ok ? P.img.sod[idx] : 0;
    uint32_t u = (uint32_t)e & (uint32_t)kIdMask;
    bool hit = ok && class_has(P, W.cls_base, u, b);
    const uint64_t it = item_of(u | W.gtag, W.cstart);
    emit(P, W, hit && (e & kFlagReport), it);
    bool keep = hit && !(e & kFlagDeadEnd) && (W.cstart + 1 < W.cend);
    if (keep && P.dedup && (e & kFlagDedup)) keep = dedup_fresh(P, W, it);
    push<Stage>(P, W, keep, it);
  }
}

// The same for every group (cross-group work items): (tagged id, group)
// pairs, each group's class base from its metadata.
template <bool Stage = false>
NGAP_DEV void seed_start_all(const KParams &P, WaveState &W) {
  const uint32_t b = P.input[W.cstart];
  for (uint32_t i = 0; i < P.img.n_xsod; i += kWave) {
    const uint32_t idx = i + W.lane;
    const bool ok = idx < P.img.n_xsod;
    int32_t e = 0;
    uint32_t g = 0;
    bool hit = false;
    if (ok) {
      e = (int32_t)P.img.xsod[2 * idx];
      g = P.img.xsod[2 * idx + 1];
      hit = class_has(P, P.img.meta[g].cls_base, (uint32_t)e & (uint32_t)kIdMask, b);
    }
    const uint64_t it = item_of(((uint32_t)e & (uint32_t)kIdMask) | (g << 22), W.cstart);
    emit(P, W, hit && (e & kFlagReport), it);
    bool keep = hit && !(e & kFlagDeadEnd) && (W.cstart + 1 < W.cend);
    if (keep && P.dedup && (e & kFlagDedup)) keep = dedup_fresh(P, W, it);
    push<Stage>(P, W, keep, it);
  }
}

// One step of every valid lane's item: test its successors on the next byte.
// Lane context of the item being expanded: group tag and the group's record
// and class bases.
struct LaneGroup {
  uint32_t gtag, rec_base, cls_base;
};

// Where expand() finds a position's chunk end: engine runs (chunks of
// chunk_len bytes, a divisibility test valid for items of any work item),
// request runs of the streaming kernel (the last-byte map), or decided at run
// time (chunk_len, else the wave's one open work item's bounds).
enum : int { kEndChunkLen = 0, kEndMap = 1, kEndRuntime = 2 };

// The step is written for few instructions, which bound it as much as its two
// dependent gathers do (with four waves a SIMD, vector instructions took two
// thirds of the SIMDs' cycles): hits are lane masks first, and reports, the
// de-duplication cache and successors beyond a lane's first are looked at only
// when some lane has one.
template <int End = kEndRuntime>
NGAP_DEV void expand(const KParams &P, WaveState &W, bool &valid, uint32_t &v,
                     uint32_t &p, int &depth, const LaneGroup &lg) {
  const uint32_t p1 = p + 1;
  // unconditional loads (index 0 stands in for idle lanes; some lane is valid,
  // so the image has a record)
  const uint32_t b = P.input[valid ? p1 : 0u];
  Rec rec = load_rec(P, valid ? lg.rec_base + v : 0u);
  const uint32_t busy = __popcll(wballot(valid));
  W.items += busy;
  // is p1 the last position of its chunk (no successors enabled after it)?
  bool last;
  if (End == kEndMap) {
    const uint32_t lw = P.last_map[valid ? p1 >> 5 : 0u];
    last = ((lw >> (p1 & 31)) & 1u) != 0u;
  } else if (End == kEndChunkLen || P.chunk_len) {
    // divisible by chunk_len = odd << div_shift: n * (odd's inverse), rotated,
    // stays small exactly for the multiples (Granlund and Montgomery)
    const uint32_t n = (p1 + 1) * P.div_inverse;
    last = __builtin_rotateright32(n, P.div_shift) <= P.div_most;
  } else {
    last = p1 + 1 >= W.cend;
  }
  // work privatization (kernel_ngap_O4.cu:115-122): a matched successor is
  // expanded by the same lane while more than active_threshold lanes are
  // busy, and otherwise queued for the idle lanes
  const bool can_priv = ((P.priv_limit < 0) | (depth < P.priv_limit)) &
                        ((int32_t)busy > P.active_threshold);
  bool has_next = false;
  uint32_t nv = 0;
  bool more = valid;
  for (;;) {
    const int32_t es[4] = {rec.ids.x, rec.ids.y, rec.ids.z, rec.ids.w};
    const uint32_t ts[4] = {rec.tests.x, rec.tests.y, rec.tests.z, rec.tests.w};
    // class words of the successors that are not decided by their test word;
    // successors fill the slots from 0 (a continuation link is in the last), so
    // the later slots are often empty in every lane, and are skipped then: tested
    // all the same, units of the plain schedule took 5.10 ms and take 4.88 (1,024
    // automata, 2 MiB, depth 2)
    bool need[4], hit[4] = {false, false, false, false}, keep[4] = {false, false, false, false};
    uint32_t cw[4] = {0, 0, 0, 0};
    bool rep = false, dup = false;
    auto fetch = [&](int s) {
      need[s] = more & (es[s] >= 0) & (ts[s] == 0u);
      if (wballot(need[s])) {
        const uint32_t u = (uint32_t)es[s] & (uint32_t)kIdMask;
        cw[s] = P.img.cls[need[s] ? (size_t)(lg.cls_base + u) * 8 + (b >> 5) : 0];
      }
    };
    auto test = [&](int s) {
      const bool in_class = ((cw[s] >> (b & 31)) & 1u) != 0;
      hit[s] = more & ((ts[s] == (b | kTestLiteral)) | (ts[s] == kTestAll) | (need[s] & in_class));
      rep |= hit[s] & ((es[s] & kFlagReport) != 0);
      keep[s] = hit[s] & ((es[s] & kFlagDeadEnd) == 0) & !last;
      dup |= keep[s] & ((es[s] & kFlagDedup) != 0);
    };
    fetch(0);
    if (wballot(more & (es[1] >= 0))) {
      fetch(1);
      if (wballot(more & (es[2] >= 0))) {
        fetch(2);
        fetch(3);
        test(2);
        test(3);
      }
      test(1);
    }
    test(0);
    if (wballot(rep)) {
#pragma unroll
      for (int s = 0; s < 4; s++)
        emit(P, W, hit[s] & ((es[s] & kFlagReport) != 0),
             item_of(((uint32_t)es[s] & (uint32_t)kIdMask) | lg.gtag, p1));
    }
    if (P.dedup && wballot(dup)) {
#pragma unroll
      for (int s = 0; s < 4; s++)
        if (keep[s] & ((es[s] & kFlagDedup) != 0))
          keep[s] = dedup_fresh(
              P, W, item_of(((uint32_t)es[s] & (uint32_t)kIdMask) | lg.gtag, p1));
    }
    bool queue[4], any = false;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const bool take = keep[s] & !has_next & can_priv;
      nv = take ? (uint32_t)es[s] & (uint32_t)kIdMask : nv;
      has_next |= take;
      queue[s] = keep[s] & !take;
      any |= queue[s];
    }
    if (wballot(any)) {
#pragma unroll
      for (int s = 0; s < 4; s++)
        push(P, W, queue[s], item_of(((uint32_t)es[s] & (uint32_t)kIdMask) | lg.gtag, p1));
    }
    // a continuation record (more than four successors)
    const int32_t e3 = es[3];
    more = more & (e3 <= -2);
    if (wballot(more) == 0) break;
    rec = load_rec(P, more ? (uint32_t)-(e3 + 2) : 0u);
  }
  // selects, not a branch: a divergent branch that joins at the caller's loop
  // end would make every counter merged there a vector
  v = has_next ? nv : v;
  p = has_next ? p1 : p;
  depth += has_next ? 1 : 0;
  valid = has_next;
}

NGAP_DEV void clear_dedup(const KParams &P, WaveState &W) {
  for (uint32_t i = W.lane; i < kDc; i += kWave) W.dc[i] = ~0ull;
  wsync();
}

// The current (group, chunk): group bases, tag and root masks in LDS.
NGAP_DEV void set_unit(const KParams &P, WaveState &W, uint32_t g, uint32_t cstart,
                       uint32_t cend) {
  const GroupMeta gm = P.img.meta[g];
  W.g = g;
  W.gtag = g << 22;
  W.rec_base = gm.rec_base;
  W.cls_base = gm.cls_base;
  W.cstart = cstart;
  W.cend = cend;
  if (W.lane < 16) W.mask1[W.lane] = P.img.mask1[g * 16 + W.lane];
  wsync();
}

// A cross-group work item: every group's roots in one window of a chunk.
NGAP_DEV void set_cross(const KParams &P, WaveState &W, uint32_t cstart, uint32_t cend) {
  W.g = kAllGroups;
  W.gtag = 0;
  W.cstart = cstart;
  W.cend = cend;
  if (W.lane < 8) W.mask1[8 + W.lane] = P.img.xmask1[W.lane];  // bytes with depth-1 reports
  wsync();
}

NGAP_DEV void begin_unit(const KParams &P, WaveState &W, uint32_t g, uint32_t cstart,
                         uint32_t cend) {
  clear_dedup(P, W);
  set_unit(P, W, g, cstart, cend);
}

NGAP_DEV void begin_cross(const KParams &P, WaveState &W, uint32_t cstart, uint32_t cend) {
  clear_dedup(P, W);
  set_cross(P, W, cstart, cend);
}

NGAP_DEV void setup_wave(WaveState &W, unsigned char *base, uint32_t wave) {
  W.rbuf = reinterpret_cast<uint64_t *>(base);
  W.dc = W.rbuf + kRbuf;
  W.sh_pref = reinterpret_cast<uint32_t *>(W.dc + kDc);
  W.sh_beg = W.sh_pref + 65;
  W.sh_pos = W.sh_beg + 64;
  W.sh_tag = W.sh_pos + 64;
  W.mask1 = W.sh_tag + 64;
  W.open = W.mask1 + 16;
  W.ring = reinterpret_cast<uint64_t *>(base + kWaveFixed);
  W.wave = wave;
  W.n_open = 0;
  W.out = nullptr;
  W.out_count = nullptr;
  W.out_cap = 0;
  W.head = W.tail = W.rn = W.spill_n = 0;
  W.lane = lane_id();
  W.overflow = false;
  W.items = 0;
}

// Runs items to completion, pulling root batches from `src` whenever the
// ring runs low.  Every loop iteration is wave-uniform.
template <bool Cross, class Src>
NGAP_DEV void drain(const KParams &P, WaveState &W, Src &src) {
  bool valid = false;
  uint32_t v = 0, p = 0;
  int depth = 0;
  LaneGroup lg{W.gtag, W.rec_base, W.cls_base};
  bool roots_left = true;
  for (;;) {
    uint32_t qn = W.tail - W.head;
    if (qn < kWave && W.spill_n > 0) {
      refill_from_spill(P, W);
      qn = W.tail - W.head;
    }
    // the next root batch runs while half the ring is still queued, so the
    // expansion steps after it find items for every idle lane
    if (qn < P.ring_cap / 2 && W.spill_n == 0 && roots_left) {
      uint32_t a, b;
      if (!src.next(W, a, b)) roots_left = false;
      else if (Cross) roots_cross(P, W, a, b);
      else roots<false, false>(P, W, a, b);
      continue;
    }
    const uint64_t idle = wballot(!valid);
    uint32_t avail = W.tail - W.head;
    uint32_t nidle = __popcll(idle);
    uint32_t take = nidle < avail ? nidle : avail;
    uint32_t r = mask_rank(idle);
    if (!valid && r < take) {
      uint64_t it = W.ring[(W.head + r) & (P.ring_cap - 1)];
      v = (uint32_t)it & (uint32_t)kIdMask;
      p = (uint32_t)(it >> 32);
      valid = true;
      depth = 0;
      if (Cross) {
        const uint32_t g = ((uint32_t)it >> 22) & 1023u;
        const uint2 base = *reinterpret_cast<const uint2 *>(&P.img.meta[g]);
        lg.gtag = g << 22;
        lg.rec_base = base.x;
        lg.cls_base = base.y;
      }
    }
    W.head += take;
    wsync();
    if (wballot(valid) == 0) {
      if (W.tail == W.head && W.spill_n == 0 && !roots_left) break;
      continue;
    }
    expand(P, W, valid, v, p, depth, lg);
  }
}

// A wave's claims of work items.  A workgroup's own items (one a row, own_item) are
// taken by its waves with an LDS counter, the others are in one queue an XCD
// (queue_item), from which a wave claims by an atomic in memory.  Such
// an atomic is a round trip of 2 us, and those of thousands of waves on one address
// take 20 ns each, one after the other: 2 MiB scanned in two items a wave took
// 0.086 ms with all claimed so (the queues' ends found by two more atomics a wave)
// and takes 0.056 with none.  So items of about the same cost (P.even) are all the
// workgroups' own up to kOwnItems a wave, which is enough to even out the waves'
// times within a workgroup, and three quarters of them above, where the rest evens
// out the workgroups' (1,024 automata, 64 MiB, 16 items a wave: 1.12 ms with all
// owned, 1.09 so).  Of other items only a wave's first is its own.
constexpr uint32_t kOwnItems = 6;
struct Claims {
  uint32_t *word;    // LDS: the workgroup's items taken; its queue is empty
  uint32_t per;      // its items
  uint32_t queues, q;
  uint32_t ahead;    // lane 0: what an early claim returned
  bool first, own, asked, dry;
  // all of the workgroup's threads; two words of LDS
  NGAP_DEV void start(const KParams &P, uint32_t *lds) {
    const uint32_t waves = P.waves_per_block, wgs = gridDim.x;
    const uint64_t all = (uint64_t)waves * wgs;
    per = P.num_tasks <= all * (P.even ? kOwnItems : 1)
              ? (P.num_tasks + wgs - 1) / wgs
              : P.even ? (uint32_t)((uint64_t)P.num_tasks * 3 / 4 / wgs) : waves;
    word = lds;
    if (threadIdx.x == 0) {
      word[0] = waves;  // a wave's first item is its own
      word[1] = 0;
    }
    __syncthreads();
    queues = min_u(kQueues, wgs);
    q = blockIdx.x % kQueues;
    ahead = 0;
    first = own = true;
    asked = false;
    dry = (uint64_t)per * wgs + q >= P.num_tasks;
  }
  // claims from the queue early
  NGAP_DEV void ask(const KParams &P, const WaveState &W) {
    if (asked | own | dry) return;
    dry = from_first(word[1]) != 0;
    if (dry) return;
    if (W.lane == 0) ahead = atomicAdd(P.task_head + q * kQueueStride, 1u);
    asked = true;
  }
  // the next work item, or P.num_tasks when there is none
  NGAP_DEV uint32_t claim(const KParams &P, const WaveState &W) {
    if (own) {
      uint32_t i = W.wave;
      if (!first) {
        i = 0;
        if (W.lane == 0) i = atomicAdd(word, 1u);
        i = from_first(i);
      }
      first = false;
      const uint64_t t = own_item(i, blockIdx.x, gridDim.x);
      if ((i < per) & (t < P.num_tasks)) return (uint32_t)t;
      own = false;
    }
    ask(P, W);
    if (!asked) return P.num_tasks;
    asked = false;
    const uint64_t t = (uint64_t)per * gridDim.x + queue_item(from_first(ahead), q, queues);
    if (t < P.num_tasks) return (uint32_t)t;
    dry = true;
    if (W.lane == 0) word[1] = 1;
    return P.num_tasks;
  }
};

// Batched schedule, engine runs: the wave's stream of work items.  A wave
// starts the next work item as soon as the current one has no positions left
// and its queue runs low, so the tail of one work item's items overlaps the
// roots of the next; at most kMaxOpen work items are open (items possibly
// queued) at a time.  next(): 0 = a root batch [a, b), 1 = wait for the open
// work items to finish, 2 = the queue is empty.
struct TaskStream {
  uint32_t cur = 0, end = 0;
  uint64_t rbase = 0;       // root pass: the work item's first root item
  bool cross = false;
  bool cross_mask = false;  // LDS holds the cross-group report mask
  Claims claims;
  template <bool RootItems, bool Gen>
  NGAP_DEV int next(const KParams &P, WaveState &W, uint32_t &a, uint32_t &b) {
    if (cur >= end) {
      if (W.n_open >= kMaxOpen) return 1;
      const uint32_t t = claims.claim(P, W);
      if (t >= P.num_tasks) return 2;
      const uint32_t ti = P.task_order ? P.task_order[t] : t;
      const Task T = Gen ? gen_task(P, ti) : P.tasks[ti];
      if (W.lane == 0) W.open[W.n_open] = ti;
      W.n_open++;
      if (RootItems) {  // the root pass wrote this work item's roots
        rbase = P.root_off[ti];
        const uint64_t cap = P.root_off[ti + 1] - rbase;
        const unsigned long long n = P.root_count[ti];
        cur = 0;
        end = (uint32_t)(n < cap ? n : cap);
        a = cur;
        b = end < kWave ? end : kWave;
        cur = b;
        return 0;
      }
      cross = T.group == kAllGroups;
      if (cross) {
        if (!cross_mask) set_cross(P, W, T.cstart, T.cend);
        W.g = kAllGroups;
        W.gtag = 0;
        W.cstart = T.cstart;
        W.cend = T.cend;
        cross_mask = true;
        if (T.flags & kTaskSeedStart) seed_start_all(P, W);
      } else {
        set_unit(P, W, T.group, T.cstart, T.cend);
        cross_mask = false;
        if (T.flags & kTaskSeedStart) {
          const GroupMeta gm = P.img.meta[T.group];
          seed_start_of_data(P, W, gm.sod_begin, gm.sod_end);
        }
      }
      cur = T.begin;
      end = T.end;
    }
    a = cur;
    // roots_cross takes two halves; the root pass's items go 64 at a time,
    // per-group roots root_batch positions at a time
    const uint32_t step = RootItems ? kWave : cross ? 2 * kWave : P.root_batch;
    b = cur + step < end ? cur + step : end;
    cur = b;
    return 0;
  }
};

// All queued items are done: the open work items are complete, and each is
// marked for the overflow fallback when the wave dropped an item since they
// opened.
NGAP_DEV void close_open(WaveState &W) {
  if (W.n_open == 0) return;
  wsync();
  if (W.overflow) {
    const KParams &P = cold_params();
    if (W.lane < W.n_open) atomicOr(&P.overflow[W.open[W.lane]], kSpillOverflow);
    if (W.lane == 0) atomicAdd(P.overflow_count, W.n_open);
  }
  W.n_open = 0;
  W.overflow = false;
  wsync();
}

// Queues root items [from, from + n) of the root pass (n <= 64).
NGAP_DEV void take_roots(const KParams &P, WaveState &W, uint64_t from, uint32_t n) {
  if (n == 0) return;
  const bool ok = W.lane < n;
  const uint64_t it = P.root_items[ok ? from + W.lane : from];
  push(P, W, ok, it);
}

// drain() over a TaskStream: items of several work items (and groups) share
// the queue, so a lane looks up its item's group bases when it takes one.
template <bool RootItems, int End, bool Gen>
NGAP_DEV void drain_stream(const KParams &P, WaveState &W, uint32_t *word) {
  TaskStream src;
  src.claims.start(P, word);
  bool valid = false;
  uint32_t v = 0, p = 0;
  int depth = 0;
  LaneGroup lg{0u, 0u, 0u};
  bool more = true;
  for (;;) {
    uint32_t qn = W.tail - W.head;
    if (qn < kWave && W.spill_n > 0) {
      refill_from_spill(P, W);
      qn = W.tail - W.head;
    }
    if (qn < P.ring_cap / 2 && W.spill_n == 0 && more) {  // as in drain()
      uint32_t a, b;
      const int st = src.template next<RootItems, Gen>(P, W, a, b);
      if (st == 0) {
        if (RootItems) take_roots(P, W, src.rbase + a, b - a);
        else if (src.cross) roots_cross(P, W, a, b);
        else roots(P, W, a, b);
        continue;
      }
      if (st == 2) more = false;
    }
    const uint64_t idle = wballot(!valid);
    const uint32_t avail = W.tail - W.head;
    const uint32_t nidle = __popcll(idle);
    const uint32_t take = nidle < avail ? nidle : avail;
    const uint32_t r = mask_rank(idle);
    if (!valid && r < take) {
      const uint64_t it = W.ring[(W.head + r) & (P.ring_cap - 1)];
      v = (uint32_t)it & (uint32_t)kIdMask;
      p = (uint32_t)(it >> 32);
      valid = true;
      depth = 0;
      const uint32_t g = ((uint32_t)it >> 22) & 1023u;
      const uint2 base = *reinterpret_cast<const uint2 *>(&P.img.meta[g]);
      lg.gtag = g << 22;
      lg.rec_base = base.x;
      lg.cls_base = base.y;
    }
    W.head += take;
    wsync();
    if (wballot(valid) == 0) {
      if (W.tail == W.head && W.spill_n == 0) {
        close_open(W);
        if (!more) break;
      }
      continue;
    }
    expand<End>(P, W, valid, v, p, depth, lg);
  }
}

// x of another lane.
NGAP_DEV uint32_t from_lane(uint32_t x, uint32_t lane) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(lane << 2), (int)x);
}

// A load at a 32-bit byte offset from a wave-uniform base.
template <class T>
NGAP_DEV T load_at(const void *base, uint32_t byte_offset) {
  return *reinterpret_cast<const T *>(static_cast<const char *>(base) + byte_offset);
}

// ---- all-group scan at memo depth 3 (k_scan) ----
// The engine's main path: every work item scans a window for all groups,
// memo depth 3, and no list of depth 1 or 2 reports in any group (patterns of
// three or more symbols), so a position's 3-gram slot holds all there is to do
// there.  A kernel of its own: without the other levels' index arrays its
// scalar state fits the scalar registers (the general kernel spills over a
// hundred of them into vector lanes, and moving them back and forth is vector
// work), and the roots need a third of the instructions.  With it, the filters and
// the present windows and claims, against one kernel for all levels without them:
// 400,000 states over 16 MiB 0.213 -> 0.120 ms, 1,024 automata over 8 MiB 0.272 ->
// 0.191, over 64 MiB 1.77 -> 1.11, eight automata of short words over 4 MiB of text
// 0.139 -> 0.100.  (The general kernel of now beside it: scan_image.)  What bounds it is
// the latency of its gathers (slot, pairs, records: 4 MiB of L2 per XCD against
// 128 MiB of slots) and, at the end of a run, of the last chains' steps.

// A 3-gram that some group's depth-3 list has, waiting for its slot: the key
// in bits 0-23, the filter bit of the byte after it in 24-28, bit 29 set when
// the 3-gram ends its chunk, the position of its last byte in the upper word.
constexpr uint32_t kKeyLast = 1u << 29;

struct ScanLds {
  uint32_t *mark;       // [kWave]
  uint64_t *keys;       // [kKeyCap], `n_keys` of them waiting
  const uint2 *bases;   // (record, class) bases of every group
  uint32_t n_keys;
};

// The 3-grams at positions [a, b), b - a <= 128, that have a list in some
// group, by the presence bitmap (2 MiB: it stays in L2, where the 128 MiB of
// slots do not).  Two neighbouring positions a lane, from one 8-byte load of
// the input (at most P.load_last, so that it stays inside the input).  The
// slots are read by whole waves of present 3-grams (take_keys).  It takes 0.83 of
// the time of a slot read at every position where the lists cover one 3-gram in 28
// (400,000 states, 16 MiB), 1.03 where they cover nearly half (1,024 automata, 64
// MiB).
NGAP_DEV void find_keys(const KParams &P, WaveState &W, ScanLds &S, uint32_t a, uint32_t b) {
  const uint32_t p = a + 2 * W.lane;
  // 3-grams end before the chunk does
  const uint32_t lim = b + 2 <= W.cend ? b : W.cend - (W.cend < 2 ? W.cend : 2);
  const uint32_t at = min_u(p, P.load_last);
  uint64_t bytes;
  __builtin_memcpy(&bytes, P.input + at, 8);
  bytes >>= 8 * min_u(p - at, 7);
  const uint32_t lo = (uint32_t)bytes, hi = (uint32_t)(bytes >> 32);
  const uint32_t key[2] = {__builtin_amdgcn_perm(hi, lo, 0x0c000102u),
                           __builtin_amdgcn_perm(hi, lo, 0x0c010203u)};
  const uint32_t next[2] = {lo >> 24, hi & 255u};
  uint32_t word[2];
#pragma unroll
  for (int h = 0; h < 2; h++) word[h] = load_at<uint32_t>(P.img.xb3, (key[h] >> 5) << 2);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const bool has = (p + h < lim) & (((word[h] >> (key[h] & 31)) & 1u) != 0);
    const uint64_t m = wballot(has);
    const uint32_t low = key[h] | (filter_bit(next[h]) << 24) |
                         (p + h + 3 >= W.cend ? kKeyLast : 0u);
    if (has) S.keys[S.n_keys + mask_rank(m)] = ((uint64_t)(p + h + 2) << 32) | low;
    wsync();
    S.n_keys += __popcll(m);
  }
}

// Roots from the slots of up to 64 waiting 3-grams, one a lane.
NGAP_DEV void take_keys(const KParams &P, WaveState &W, ScanLds &S) {
  const uint32_t count = min_u(S.n_keys, kWave);
  S.n_keys -= count;
  const bool have = W.lane < count;
  const uint64_t entry = S.keys[S.n_keys + (have ? W.lane : 0u)];
  const uint32_t key = (uint32_t)entry, pos = (uint32_t)(entry >> 32);
  const uint2 slot = load_at<uint2>(P.img.xs3, (key & 0xFFFFFFu) << 3);
  const uint32_t bit = (key >> 24) & 31;
  // an inline state: the one entry, in the slot itself
  const bool inl = have & ((int32_t)slot.y < 0);
  {
    bool keep = inl & ((slot.x & (uint32_t)kFlagDeadEnd) == 0) & ((key & kKeyLast) == 0);
    const uint64_t it = item_of((slot.x & (uint32_t)kIdMask) | (slot.y << 22), pos);
    if (NGAP_SELDOM(wballot(inl & ((slot.x & (uint32_t)(kFlagReport | kFlagDedup)) != 0)))) {
      emit(P, W, inl & ((slot.x & (uint32_t)kFlagReport) != 0), it);
      if (P.dedup && (keep & ((slot.x & (uint32_t)kFlagDedup) != 0)))
        keep = dedup_fresh(P, W, it);
      wsync();
    }
    const bool pass = keep & (((slot_filter(slot.x, slot.y) >> bit) & 1u) != 0);
    W.items += __popcll(wballot(keep & !pass));
    push(P, W, pass, it);
  }
  // the other slots' pairs, spread over the wave: owners mark where their
  // entries start and a running maximum finds each entry's owner
  const uint32_t cnt = (have & !inl) ? slot.y : 0u;
  if (wballot(cnt != 0) == 0) return;
  const uint32_t incl = dpp_scan(cnt, [](uint32_t x, uint32_t y) { return x + y; });
  const uint32_t excl = incl - cnt, total = from_last(incl);
  // entry j of the wave's flat index space is its owner's pair j + at
  const uint32_t at = slot.x - excl;
  uint32_t carry = 0;  // owner of the entries before this round's first mark, plus 1
  for (uint32_t base = 0; base < total; base += kWave) {
    S.mark[W.lane] = W.lane == 0 ? carry : 0u;
    wsync();
    if ((cnt != 0) & (excl - base < kWave)) S.mark[excl - base] = W.lane + 1;
    wsync();
    const uint32_t own =
        dpp_scan(S.mark[W.lane], [](uint32_t x, uint32_t y) { return x > y ? x : y; });
    carry = from_last(own);
    const uint32_t j = base + W.lane;
    const bool ok = j < total;
    const uint32_t wat = from_lane(at, own - 1), wkey = from_lane(key, own - 1),
                   wpos = from_lane(pos, own - 1);
    const uint32_t idx = ok ? j + wat : 0u;
    const uint2 e = reinterpret_cast<const uint2 *>(P.img.xp3)[idx];
    const uint32_t f = P.img.xf3[idx];
    const uint64_t it = item_of((e.x & (uint32_t)kIdMask) | (e.y << 22), wpos);
    bool k = ok & ((e.x & (uint32_t)kFlagDeadEnd) == 0) & ((wkey & kKeyLast) == 0);
    if (NGAP_SELDOM(wballot(ok & ((e.x & (uint32_t)(kFlagReport | kFlagDedup)) != 0)))) {
      emit(P, W, ok & ((e.x & (uint32_t)kFlagReport) != 0), it);
      if (P.dedup && (k & ((e.x & (uint32_t)kFlagDedup) != 0))) k = dedup_fresh(P, W, it);
      wsync();
    }
    const bool pass = k & (((f >> ((wkey >> 24) & 31)) & 1u) != 0);
    W.items += __popcll(wballot(k & !pass));
    push(P, W, pass, it);
  }
  wsync();
}

// The item a lane expands: its position (kNoItem: none), byte offsets of its
// state's record and of its group's first record and class, its group's tag.
struct ScanItem {
  uint32_t pos, rec, rec_base, cls_base, gtag;
};
constexpr uint32_t kNoItem = ~0u;  // (+ 1 = 0: an idle lane's loads hit position and record 0)

// expand() for k_scan: the same step with 32-bit byte offsets (the image's
// records and classes are below 4 GiB each, scan_image).  A chain of steps is
// bound by the instructions of each and above all by its branches: a step of
// a lone chain over random states took 1,050 ns in the general kernel's first
// form and takes 580 here, with 60,000 states in the cache.  So the common step
// has few branches: one to skip the slots that no lane fills, one to skip everything that
// most steps do not have (a report, a state with several predecessors, a second
// matched successor, a continuation record).
NGAP_DEV void expand_scan(const KParams &P, WaveState &W, ScanItem &I, int &depth) {
  const bool valid = I.pos != kNoItem;
  const uint32_t p1 = I.pos + 1;
  const uint32_t b = load_at<uint8_t>(P.input, p1);
  int4 ids = load_at<int4>(P.img.succ4, I.rec);
  uint4 tests = load_at<uint4>(P.img.succ4, I.rec + 16);
  const uint32_t busy = __popcll(wballot(valid));
  W.items += busy;
  const uint32_t n = (p1 + 1) * P.div_inverse;
  const bool last = __builtin_rotateright32(n, P.div_shift) <= P.div_most;
  const bool can_priv = ((P.priv_limit < 0) | (depth < P.priv_limit)) &
                        ((int32_t)busy > P.active_threshold);
  const uint32_t lit = b | kTestLiteral;
  const uint32_t cls = I.cls_base + ((b >> 5) << 2);
  bool has_next = false;
  uint32_t nv = 0;
  bool more = valid;
  for (;;) {
    const int32_t es[4] = {ids.x, ids.y, ids.z, ids.w};
    const uint32_t ts[4] = {tests.x, tests.y, tests.z, tests.w};
    bool need[4], hit[4] = {false, false, false, false}, keep[4];
    uint32_t cw[4];
    auto fetch = [&](int s) {
      need[s] = more & (es[s] >= 0) & (ts[s] == 0u);
      cw[s] = load_at<uint32_t>(
          P.img.cls, need[s] ? cls + (((uint32_t)es[s] & (uint32_t)kIdMask) << 5) : 0u);
    };
    auto test = [&](int s) {
      hit[s] = (more & ((ts[s] == lit) | (ts[s] == kTestAll))) |
               (need[s] & (((cw[s] >> (b & 31)) & 1u) != 0));
    };
    // successors fill the slots from 0 (a continuation link is in the last)
    fetch(0);
    uint32_t all = 0;  // the hit successors' tags together
    if (wballot(more & (es[1] >= 0))) {
      fetch(1);
      if (wballot(more & (es[2] >= 0))) {
        fetch(2);
        fetch(3);
        test(2);
        test(3);
        all = (hit[2] ? (uint32_t)es[2] : 0u) | (hit[3] ? (uint32_t)es[3] : 0u);
      }
      test(1);
      all |= hit[1] ? (uint32_t)es[1] : 0u;
    }
    test(0);
    all |= hit[0] ? (uint32_t)es[0] : 0u;
    bool any = false, several = false;
    uint32_t first = 0;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      keep[s] = hit[s] & ((es[s] & kFlagDeadEnd) == 0) & !last;
      several |= keep[s] & any;
      first = (keep[s] & !any) ? (uint32_t)es[s] : first;
      any |= keep[s];
    }
    if (NGAP_MOSTLY(wballot(((all & (uint32_t)(kFlagReport | kFlagDedup)) != 0) | several |
                            (any & (has_next | !can_priv)) | (more & (es[3] <= -2))) == 0)) {
      nv = any ? first : nv;
      has_next |= any;
      break;
    }
    if (wballot((all & (uint32_t)kFlagReport) != 0)) {
#pragma unroll
      for (int s = 0; s < 4; s++)
        emit(P, W, hit[s] & ((es[s] & kFlagReport) != 0),
             item_of(((uint32_t)es[s] & (uint32_t)kIdMask) | I.gtag, p1));
    }
    if (P.dedup && wballot((all & (uint32_t)kFlagDedup) != 0)) {
#pragma unroll
      for (int s = 0; s < 4; s++)
        if (keep[s] & ((es[s] & kFlagDedup) != 0))
          keep[s] =
              dedup_fresh(P, W, item_of(((uint32_t)es[s] & (uint32_t)kIdMask) | I.gtag, p1));
      wsync();
    }
    bool queue[4];
    any = false;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const bool take = keep[s] & !has_next & can_priv;
      nv = take ? (uint32_t)es[s] : nv;
      has_next |= take;
      queue[s] = keep[s] & !take;
      any |= queue[s];
    }
    if (wballot(any)) {
#pragma unroll
      for (int s = 0; s < 4; s++)
        push(P, W, queue[s], item_of(((uint32_t)es[s] & (uint32_t)kIdMask) | I.gtag, p1));
    }
    // a continuation record (more than four successors)
    more &= es[3] <= -2;
    if (wballot(more) == 0) break;
    const uint32_t link = more ? (uint32_t)-(es[3] + 2) << 5 : 0u;
    ids = load_at<int4>(P.img.succ4, link);
    tests = load_at<uint4>(P.img.succ4, link + 16);
  }
  I.pos = has_next ? p1 : kNoItem;
  I.rec = has_next ? I.rec_base + ((nv & (uint32_t)kIdMask) << 5) : 0u;
  depth += 1;
}

template <bool Gen>
__global__ void __launch_bounds__(kBlockThreads) k_scan(KParams P) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t wave = from_first(threadIdx.x / kWave);
  uint2 *bases = reinterpret_cast<uint2 *>(lds + 16);
  for (uint32_t g = threadIdx.x; g < P.num_groups; g += kBlockThreads)
    bases[g] = *reinterpret_cast<const uint2 *>(&P.img.meta[g]);
  WaveState W;
  unsigned char *mine = lds + 16 + scan_table_bytes(P.num_groups) +
                        wave * scan_wave_bytes(P.ring_cap);
  setup_wave(W, mine, wave);
  W.ring = reinterpret_cast<uint64_t *>(mine + kScanFixed);
  ScanLds S;
  S.mark = reinterpret_cast<uint32_t *>(W.dc + kDc);
  S.bases = bases;
  S.keys = reinterpret_cast<uint64_t *>(S.mark + kWave);
  S.n_keys = 0;
  W.open = reinterpret_cast<uint32_t *>(S.keys + kKeyCap);
  clear_dedup(P, W);

  Claims claims;
  claims.start(P, reinterpret_cast<uint32_t *>(lds));
  uint32_t cur = 0, end = 0;
  bool more = true;
  ScanItem I = {};
  I.pos = kNoItem;
  int depth = 0;
  for (;;) {
    // Below `low` queued items something comes before the next expansion:
    // spilled items come back; else, while half the ring is still queued (so
    // that the expansions after it find items for every idle lane), roots: of
    // a wave's width of waiting 3-grams, or of what is left of them when no
    // position can be searched any more.
    const uint32_t qn = W.tail - W.head;
    const bool search = (cur < end) | (more & (W.n_open < kMaxOpen));
    const uint32_t low = W.spill_n ? kWave : (search | (S.n_keys != 0)) ? P.ring_cap / 2 : 0u;
    if (qn < low) {
      if (NGAP_SELDOM(W.spill_n)) {
        refill_from_spill(P, W);
        continue;
      }
      if ((S.n_keys >= kWave) | !search) {
        take_keys(P, W, S);
        continue;
      }
      if (NGAP_SELDOM(cur >= end)) {
        const KParams &Q = cold_params();
        const uint32_t t = claims.claim(Q, W);
        if (t >= Q.num_tasks) {
          more = false;
          continue;
        }
        const Task T = Gen ? gen_task(Q, t) : Q.tasks[t];
        if (W.lane == 0) W.open[W.n_open] = t;
        W.n_open++;
        W.cstart = T.cstart;
        W.cend = T.cend;
        if ((T.flags & kTaskSeedStart) && Q.img.n_xsod) seed_start_all(Q, W);
        cur = T.begin;
        end = T.end;
      }
      const uint32_t stop = min_u(cur + 2 * kWave, end);
      find_keys(P, W, S, cur, stop);
      cur = stop;
      // the next work item is claimed with one step of this one left
      if (end - cur <= 2 * kWave) claims.ask(cold_params(), W);
      continue;
    }
    const uint64_t idle = wballot(I.pos == kNoItem);
    const uint32_t take = min_u(__popcll(idle), qn);
    if (take) {
      const uint32_t r = mask_rank(idle);
      if ((I.pos == kNoItem) & (r < take)) {
        const uint64_t it = W.ring[(W.head + r) & (P.ring_cap - 1)];
        const uint32_t tagged = (uint32_t)it;
        const uint2 base = S.bases[tagged >> 22];
        I.pos = (uint32_t)(it >> 32);
        I.gtag = tagged & ~(uint32_t)kIdMask;
        I.rec_base = base.x << 5;
        I.cls_base = base.y << 5;
        I.rec = I.rec_base + ((tagged & (uint32_t)kIdMask) << 5);
        depth = 0;
      }
      wsync();
      W.head += take;
    } else if (NGAP_SELDOM(idle == ~0ull)) {  // nothing queued, nothing in the lanes
      close_open(W);
      if (!more) break;
      continue;
    }
    expand_scan(P, W, I, depth);
  }
  flush_reports(W);
  if (W.lane == 0) add_items(W.items);
}

// Plain schedule: the cursor over a (group, chunk) unit shared by the block's
// waves (the reference's one-block-per-unit decomposition, ngap.cu:1507).
struct SharedCursor {
  uint32_t *cursor;
  uint32_t end, batch;
  NGAP_DEV bool next(const WaveState &W, uint32_t &a, uint32_t &b) {
    uint32_t x = 0;
    if (W.lane == 0) x = atomicAdd(cursor, batch);
    x = from_first(x);
    if (x >= end) return false;
    a = x;
    b = x + batch < end ? x + batch : end;
    return true;
  }
};

// Batched schedule: a wave walks its own work item in 64-position steps.
struct LocalCursor {
  uint32_t cur, end;
  NGAP_DEV bool next(const WaveState &W, uint32_t &a, uint32_t &b) {
    if (cur >= end) return false;
    a = cur;
    b = cur + kWave < end ? cur + kWave : end;
    cur = b;
    return true;
  }
};

// A unit's waves share its cursor, so their number is free (run_plain).
__global__ void __launch_bounds__(kPlainWaves * kWave) k_plain(KParams P) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t wave = from_first(threadIdx.x / kWave);
  const uint32_t unit = blockIdx.x;
  const uint32_t g = unit % P.num_groups, c = unit / P.num_groups;
  uint32_t *cursor = reinterpret_cast<uint32_t *>(lds);
  const uint32_t wbytes = wave_lds_bytes(P.ring_cap);
  WaveState W;
  setup_wave(W, lds + 16 + wave * wbytes, wave);
  begin_unit(P, W, g, c * P.chunk_len, (c + 1) * P.chunk_len);
  if (threadIdx.x == 0) *cursor = W.cstart;
  __syncthreads();
  if (wave == 0 && (c == 0 || P.is_dup)) {
    const GroupMeta gm = P.img.meta[g];
    seed_start_of_data(P, W, gm.sod_begin, gm.sod_end);
  }
  SharedCursor src{cursor, W.cend, P.root_batch};
  drain<false>(P, W, src);
  flush_reports(W);
  if (W.lane == 0) {
    if (W.overflow && atomicOr(&P.overflow[unit], 1u) == 0u) atomicAdd(P.overflow_count, 1u);
    add_items(W.items);
  }
}

__global__ void __launch_bounds__(kBlockThreads) k_batched(KParams P) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t wave = from_first(threadIdx.x / kWave);
  const uint32_t wbytes = wave_lds_bytes(P.ring_cap);
  WaveState W;
  setup_wave(W, lds + 16 + wave * wbytes, wave);
  Claims claims;
  claims.start(P, reinterpret_cast<uint32_t *>(lds));
  for (;;) {
    const uint32_t t = claims.claim(P, W);
    if (t >= P.num_tasks) break;
    const uint32_t ti = P.task_order ? P.task_order[t] : t;
    const Task T = P.tasks[ti];
    W.overflow = false;
    const unsigned long long items0 = W.items;
    LocalCursor src{T.begin, T.end};
    if (T.group == kAllGroups) {
      begin_cross(P, W, T.cstart, T.cend);
      if (T.flags & kTaskSeedStart) seed_start_all(P, W);
      drain<true>(P, W, src);
    } else {
      begin_unit(P, W, T.group, T.cstart, T.cend);
      if (T.flags & kTaskSeedStart) {
        const GroupMeta gm = P.img.meta[T.group];
        seed_start_of_data(P, W, gm.sod_begin, gm.sod_end);
      }
      drain<false>(P, W, src);
    }
    if (W.lane == 0) {
      if (W.overflow) {
        P.overflow[ti] = 1u;
        atomicAdd(P.overflow_count, 1u);
      }
      if (P.task_items) P.task_items[ti] = W.items - items0;
    }
  }
  flush_reports(W);
  if (W.lane == 0) add_items(W.items);
}

// The batched engine without per-work-item traces: each wave overlaps its
// work items (drain_stream).  Kernels of their own, so their registers are
// not sized for the per-item path: engine runs (End = kEndChunkLen, work
// items from P.tasks), request runs (kEndMap) and engine runs whose work
// items are generated from their index (Gen).
template <int End, bool Gen>
__global__ void __launch_bounds__(kBlockThreads) k_batched_stream(KParams P) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t wave = from_first(threadIdx.x / kWave);
  const uint32_t wbytes = wave_lds_bytes(P.ring_cap);
  WaveState W;
  setup_wave(W, lds + 16 + wave * wbytes, wave);
  clear_dedup(P, W);
  drain_stream<false, End, Gen>(P, W, reinterpret_cast<uint32_t *>(lds));
  flush_reports(W);
  if (W.lane == 0) add_items(W.items);
}

// The streaming kernel after a root pass (k_roots): its work items' roots
// are read from root_items, so it holds only the expansion's registers.
__global__ void __launch_bounds__(kBlockThreads) k_expand(KParams P) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t wave = from_first(threadIdx.x / kWave);
  const uint32_t wbytes = wave_lds_bytes(P.ring_cap);
  WaveState W;
  setup_wave(W, lds + 16 + wave * wbytes, wave);
  clear_dedup(P, W);
  drain_stream<true, kEndChunkLen, false>(P, W, reinterpret_cast<uint32_t *>(lds));
  flush_reports(W);
  if (W.lane == 0) add_items(W.items);
}

// Root pass of an engine run: one wave per piece of a work item (a non-
// persistent grid, so the gathers of many waves overlap).  The piece's roots
// (and start-of-data seeds) are staged in the wave's LDS ring and appended
// to the work item's area of root_items; their reports go out at once.
// k_batched_stream then expands the items.
__global__ void __launch_bounds__(kBlockThreads) k_roots(KParams P) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t wave = from_first(threadIdx.x / kWave);
  const uint32_t piece = blockIdx.x * P.waves_per_block + wave;
  if (piece >= P.num_pieces) return;  // wave-uniform; no block barrier follows
  const uint32_t wbytes = wave_lds_bytes(P.ring_cap);
  WaveState W;
  setup_wave(W, lds + 16 + wave * wbytes, wave);
  const RootPiece R = P.pieces[piece];
  const Task T = P.tasks[R.task];
  const uint64_t o0 = P.root_off[R.task];
  W.out = P.root_items + o0;
  W.out_cap = P.root_off[R.task + 1] - o0;
  W.out_count = P.root_count + R.task;
  if (T.group == kAllGroups) {
    begin_cross(P, W, T.cstart, T.cend);
    if (R.flags & kTaskSeedStart) seed_start_all<true>(P, W);
    for (uint32_t a = R.begin; a < R.end; a += 2 * kWave)
      roots_cross<true>(P, W, a, min_u(a + 2 * kWave, R.end));
  } else {
    begin_unit(P, W, T.group, T.cstart, T.cend);
    if (R.flags & kTaskSeedStart) {
      const GroupMeta gm = P.img.meta[T.group];
      seed_start_of_data<true>(P, W, gm.sod_begin, gm.sod_end);
    }
    for (uint32_t a = R.begin; a < R.end; a += kWave)
      roots<true>(P, W, a, min_u(a + kWave, R.end));
  }
  flush_stage(P, W);
  flush_reports(W);
  if (W.lane == 0 && W.items) add_items(W.items);  // the filtered ones
  if (W.lane == 0 && W.overflow && atomicOr(&P.overflow[R.task], kRootOverflow) == 0u)
    atomicAdd(P.overflow_count, 1u);
}

// blockinggroups (the reference's BAP baseline, kernel_ngap_O0.cu:7-126): one
// workgroup per (group, chunk) unit advances the set of states matched at
// position p to those matched at p + 1 in lock step, with a block barrier per
// input byte.  The frontier lives in a per-unit HBM buffer (two halves of
// P.spill_cap states); appends are compacted per wave.
NGAP_DEV void block_append(const KParams &P, WaveState &W, uint32_t *count, uint32_t *buf,
                           bool pred, uint32_t u) {
  const uint64_t m = wballot(pred);
  if (m == 0) return;
  const uint32_t cnt = __popcll(m);
  uint32_t base = 0;
  if (W.lane == 0) base = atomicAdd(count, cnt);
  base = from_first(base);
  const uint32_t slot = base + mask_rank(m);
  if (pred && slot < P.spill_cap) buf[slot] = u;
  // the wave's flag, whichever lane lost its state (lane 0 reports it)
  if (base + cnt > P.spill_cap) W.overflow = true;
}

__global__ void __launch_bounds__(kBlockThreads) k_blocking(KParams P) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t wave = from_first(threadIdx.x / kWave);
  const uint32_t unit = blockIdx.x;
  const uint32_t g = unit % P.num_groups, c = unit / P.num_groups;
  uint32_t *count = reinterpret_cast<uint32_t *>(lds);  // [0] current, [1] next
  const uint32_t wbytes = wave_lds_bytes(P.ring_cap);
  WaveState W;
  setup_wave(W, lds + 16 + wave * wbytes, wave);
  begin_unit(P, W, g, c * P.chunk_len, (c + 1) * P.chunk_len);
  uint32_t *front = reinterpret_cast<uint32_t *>(P.spill) + (size_t)unit * 2 * P.spill_cap;
  const GroupMeta gm = P.img.meta[g];
  const bool seed = c == 0 || P.is_dup;
  if (threadIdx.x == 0) count[0] = count[1] = 0;
  __syncthreads();
  // position cstart: matched start-of-data and all-input states
  {
    uint32_t *cur = front;
    const uint32_t b = P.input[W.cstart];
    for (uint32_t i = gm.sod_begin + wave * kWave; seed && i < gm.sod_end; i += kBlockThreads) {
      const uint32_t idx = i + W.lane;
      const bool ok = idx < gm.sod_end;
      const int32_t e = ok ? P.img.sod[idx] : 0;
      const uint32_t u = (uint32_t)e & (uint32_t)kIdMask;
      const bool hit = ok && class_has(P, W.cls_base, u, b);
      emit(P, W, hit && (e & kFlagReport), ((uint64_t)W.cstart << 32) | u | W.gtag);
      block_append(P, W, &count[0], cur, hit && !(e & kFlagDeadEnd), u);
    }
    const uint32_t li = g * 256u + b;
    const uint32_t lb = P.img.beg[0][li], le = P.img.beg[0][li + 1];
    for (uint32_t i = lb + wave * kWave; i < le; i += kBlockThreads) {
      const uint32_t idx = i + W.lane;
      const bool ok = idx < le;
      const int32_t e = ok ? P.img.list[0][idx] : 0;
      const uint32_t u = (uint32_t)e & (uint32_t)kIdMask;
      emit(P, W, ok && (e & kFlagReport), ((uint64_t)W.cstart << 32) | u | W.gtag);
      block_append(P, W, &count[0], cur, ok && !(e & kFlagDeadEnd), u);
    }
  }
  __syncthreads();
  for (uint32_t p = W.cstart; p + 1 < W.cend; p++) {
    const uint32_t sel = (p - W.cstart) & 1u;
    uint32_t *cur = front + sel * P.spill_cap;
    uint32_t *nxt = front + (sel ^ 1u) * P.spill_cap;
    uint32_t *ncount = &count[sel ^ 1u];
    const uint32_t n = min(count[sel], P.spill_cap);
    const uint32_t p1 = p + 1;
    const uint32_t b = P.input[p1];
    // successors of the matched states, tested on input[p + 1]
    for (uint32_t i = wave * kWave; i < n; i += kBlockThreads) {
      const uint32_t idx = i + W.lane;
      bool more = idx < n;
      Rec rec = empty_rec();
      if (more) rec = load_rec(P, W.rec_base + cur[idx]);
      while (wballot(more)) {
        int32_t link = -1;
        const int32_t es[4] = {rec.ids.x, rec.ids.y, rec.ids.z, rec.ids.w};
        const uint32_t ts[4] = {rec.tests.x, rec.tests.y, rec.tests.z, rec.tests.w};
#pragma unroll
        for (int s2 = 0; s2 < 4; s2++) {
          const int32_t e = es[s2];
          if (more && e <= -2) link = -(e + 2);
          const uint32_t u = (uint32_t)e & (uint32_t)kIdMask;
          const bool hit =
              test_hit(more, e, ts[s2], test_word(P, W.cls_base, more, e, ts[s2], b), b);
          emit(P, W, hit && (e & kFlagReport), item_of(u | W.gtag, p1));
          bool keep = hit && !(e & kFlagDeadEnd);
          if (keep && P.dedup && (e & kFlagDedup)) keep = dedup_fresh(P, W, item_of(u | W.gtag, p1));
          block_append(P, W, ncount, nxt, keep, u);
        }
        more = more && link >= 0;
        if (more) rec = load_rec(P, (uint32_t)link);
      }
    }
    // all-input states matched at p + 1
    const uint32_t li = g * 256u + b;
    const uint32_t lb = P.img.beg[0][li], le = P.img.beg[0][li + 1];
    for (uint32_t i = lb + wave * kWave; i < le; i += kBlockThreads) {
      const uint32_t idx = i + W.lane;
      const bool ok = idx < le;
      const int32_t e = ok ? P.img.list[0][idx] : 0;
      const uint32_t u = (uint32_t)e & (uint32_t)kIdMask;
      emit(P, W, ok && (e & kFlagReport), ((uint64_t)p1 << 32) | u | W.gtag);
      block_append(P, W, ncount, nxt, ok && !(e & kFlagDeadEnd), u);
    }
    if (wave == 0) W.items += n;
    __syncthreads();
    if (threadIdx.x == 0) count[sel] = 0;
    __syncthreads();
  }
  flush_reports(W);
  if (W.lane == 0) {
    if (W.overflow && atomicOr(&P.overflow[unit], 1u) == 0u) atomicAdd(P.overflow_count, 1u);
    add_items(W.items);
  }
}

// Clears the per-run counters with a kernel (graph-capture friendly).  A
// re-run of overflowed work items keeps the report count (keep_reports).
__global__ void k_reset(unsigned long long *report_count, unsigned long long *items,
                        uint32_t *task_head, uint32_t *overflow, uint32_t n_overflow,
                        uint32_t *overflow_count, int keep_reports,
                        unsigned long long *root_count) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    if (!keep_reports) *report_count = 0;
    for (uint32_t k = 0; k < kItemLanes; k++) items[k * kItemStride] = 0;
    for (uint32_t k = 0; k < kQueues; k++) task_head[k * kQueueStride] = 0;
    *overflow_count = 0;
  }
  for (; i < n_overflow; i += gridDim.x * blockDim.x) {
    overflow[i] = 0;
    if (root_count) root_count[i] = 0;
  }
}

// Ends a run: its counters to pinned memory (to[0] reports, to[1] items, the
// lanes summed, to[3] overflowed work items), and back to zero, so that the next
// run needs no k_reset, unless work items overflowed (their re-run goes on with the
// counts).  One wave.  A run of 25 us of matching took 49.5 with k_reset before
// it and a copy behind it, and takes 44.5.
__global__ void k_finish(unsigned long long *counters, unsigned long long *to) {
  const uint32_t lane = threadIdx.x;
  unsigned long long *items = counters + kItemsWord + lane % kItemLanes * kItemStride;
  uint32_t *head = reinterpret_cast<uint32_t *>(counters + 16) + lane % kQueues * kQueueStride;
  const unsigned long long reports = counters[0];
  const uint32_t over = (uint32_t)counters[3];
  unsigned long long n = lane < kItemLanes ? *items : 0;
  for (uint32_t d = kItemLanes / 2; d; d /= 2) n += __shfl_down(n, d);
  if (lane == 0) {
    to[0] = reports;
    to[1] = n;
    to[2] = 0;
    to[3] = over;
  }
  if (over) return;
  if (lane < kItemLanes) *items = 0;
  if (lane < kQueues) *head = 0;
  if (lane == 0) counters[0] = 0;
}

hipError_t launch_finish(hipStream_t s, unsigned long long *counters, unsigned long long *to) {
  static_assert(kItemLanes <= kWave && kQueues <= kWave, "one wave");
  hipLaunchKernelGGL(k_finish, dim3(1), dim3(kWave), 0, s, counters, to);
  return hipGetLastError();
}

// Host-side launch wrappers (this translation unit owns the kernels).
hipError_t launch_reset(hipStream_t s, unsigned long long *rc, unsigned long long *items,
                        uint32_t *head, uint32_t *ovf, uint32_t n, uint32_t *ovf_count,
                        int keep_reports, unsigned long long *root_count) {
  uint32_t blocks = (n + 255) / 256;
  if (blocks == 0) blocks = 1;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(k_reset, dim3(blocks), dim3(256), 0, s, rc, items, head, ovf, n,
                     ovf_count, keep_reports, root_count);
  return hipGetLastError();
}

hipError_t launch_plain(hipStream_t s, const KParams &P, uint32_t units, uint32_t lds) {
  hipLaunchKernelGGL(k_plain, dim3(units), dim3(P.waves_per_block * kWave), lds, s, P);
  return hipGetLastError();
}

hipError_t launch_blocking(hipStream_t s, const KParams &P, uint32_t units, uint32_t lds) {
  hipLaunchKernelGGL(k_blocking, dim3(units), dim3(kBlockThreads), lds, s, P);
  return hipGetLastError();
}

hipError_t launch_roots(hipStream_t s, const KParams &P, uint32_t lds) {
  const uint32_t blocks = (P.num_pieces + P.waves_per_block - 1) / P.waves_per_block;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_roots, dim3(blocks), dim3(kBlockThreads), lds, s, P);
  return hipGetLastError();
}

// The kernel of each batched kind (batched_kind).
static const void *batched_kernel(int kind) {
  switch (kind) {
    case 1: return reinterpret_cast<const void *>(k_batched_stream<kEndChunkLen, false>);
    case 2: return reinterpret_cast<const void *>(k_expand);
    case 3: return reinterpret_cast<const void *>(k_batched_stream<kEndMap, false>);
    case 4: return reinterpret_cast<const void *>(k_batched_stream<kEndChunkLen, true>);
    case 5: return reinterpret_cast<const void *>(k_scan<false>);
    case 6: return reinterpret_cast<const void *>(k_scan<true>);
    default: return reinterpret_cast<const void *>(k_batched);
  }
}

hipError_t launch_batched(hipStream_t s, const KParams &P, uint32_t blocks, uint32_t lds) {
  const int kind = batched_kind(P);
  switch (kind) {
    case 1:
      hipLaunchKernelGGL((k_batched_stream<kEndChunkLen, false>), dim3(blocks),
                         dim3(kBlockThreads), lds, s, P);
      break;
    case 2:
      hipLaunchKernelGGL(k_expand, dim3(blocks), dim3(kBlockThreads), lds, s, P);
      break;
    case 3:
      hipLaunchKernelGGL((k_batched_stream<kEndMap, false>), dim3(blocks), dim3(kBlockThreads),
                         lds, s, P);
      break;
    case 4:
      hipLaunchKernelGGL((k_batched_stream<kEndChunkLen, true>), dim3(blocks),
                         dim3(kBlockThreads), lds, s, P);
      break;
    case 5:
      hipLaunchKernelGGL(k_scan<false>, dim3(blocks), dim3(kBlockThreads), lds, s, P);
      break;
    case 6:
      hipLaunchKernelGGL(k_scan<true>, dim3(blocks), dim3(kBlockThreads), lds, s, P);
      break;
    default:
      hipLaunchKernelGGL(k_batched, dim3(blocks), dim3(kBlockThreads), lds, s, P);
  }
  return hipGetLastError();
}

hipError_t batched_occupancy(int *blocks_per_cu, uint32_t lds, int kind) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, batched_kernel(kind),
                                                      kBlockThreads, lds);
}

hipError_t set_lds_limit(uint32_t lds) {
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_plain),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_blocking),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  for (int kind = 1; kind <= kBatchedKinds - 1; kind++) {
    e = hipFuncSetAttribute(batched_kernel(kind), hipFuncAttributeMaxDynamicSharedMemorySize,
                            lds);
    if (e != hipSuccess) return e;
  }
  e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_roots),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_expand),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute(reinterpret_cast<const void *>(k_batched),
                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
}

}  // namespace ngapamd
