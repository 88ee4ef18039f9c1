// ngap_run_noalloc: an engine run that allocates no device memory, for
// callers that cannot call hipMalloc (code under stream capture, tight
// serving loops, harnesses that forbid allocation).
//
// The run's scratch memory (counters and work-queue heads, per-work-item
// overflow flags, worklist spill areas) lives in the file-scope device array
// `scratch` below, whose device address is looked up once per device when an
// engine is created (ngap_noalloc_attach).  The caller passes the input and
// the report buffer, both in device memory; the work items are generated by
// the kernel from their index, so nothing is uploaded.  Every run on a device
// shares that device's array: runs that overlap on one device race, and the
// counters and flags are cleared by a kernel at the start of every run.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "runtime.h"
#include "c_guard.h"

namespace ngapamd {

// Layout of the scratch array: the run counters (kCounterBytes of them: the
// report count, the queue heads and the item-count lanes, cleared by the reset
// kernel) then the per-work-item overflow flags,
// then the worklist spill areas.
constexpr uint64_t kScratchCounters = 8192;
constexpr uint64_t kScratchFlags = 4ull << 20;  // 1M work items
constexpr uint64_t kScratchSpill = 44ull << 20;
constexpr uint64_t kScratchBytes = kScratchCounters + kScratchFlags + kScratchSpill;

static_assert(kCounterBytes <= kScratchCounters, "run counters beyond the counter area");

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_mu;
void *g_ptr[kMaxDevices] = {nullptr};  // the array's address on each device
}  // namespace

// With `device` current: looks up this device's copy of the scratch array
// (once per device).
int noalloc_attach(int device, void **out) {
  if (device < 0 || device >= kMaxDevices)
    return ngap_fail(NGAP_ERR_INVALID, "device ordinal beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_mu);
  if (!g_ptr[device]) {
    void *p = nullptr;
    HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return ngap_fail(NGAP_ERR_DEVICE, "scratch array has no device address");
    g_ptr[device] = p;
  }
  *out = g_ptr[device];
  return NGAP_OK;
}

}  // namespace ngapamd

using namespace ngapamd;

extern "C" int ngap_run_noalloc(ngap_engine *eng, const ngap_run_opts *opts,
                                const uint8_t *d_input, uint64_t chunk_len, uint32_t num_seg,
                                uint64_t *d_reports, uint64_t report_cap,
                                ngap_run_stats *st) {
  return ngapamd::c_guard([&]() -> int {
    if (!eng || !opts || !d_input || !d_reports)
      return ngap_fail(NGAP_ERR_INVALID, "NULL argument");
    if (st) memset(st, 0, sizeof *st);
    const ngap_run_opts &o = *opts;
    if (!eng->loaded) return ngap_fail(NGAP_ERR_STATE, "no groups loaded");
    if (!eng->scratch) return ngap_fail(NGAP_ERR_STATE, "scratch array not attached");
    if (chunk_len == 0 || num_seg == 0) return ngap_fail(NGAP_ERR_INVALID, "empty input");
    if (chunk_len * num_seg >= (1ull << 32) - (1ull << 20))
      return ngap_fail(NGAP_ERR_INVALID,
                       "input offsets are 32-bit: total input must be < 4 GiB - 1 MiB");
    if (o.report_off) return ngap_fail(NGAP_ERR_INVALID, "report_off: use ngap_run");
    HIP_TRY(hipSetDevice(eng->device));
    Mapping mp;
    std::string err;
    if (!map_algorithm(o.algorithm, o.precompute_depth, eng->img.memo_depth, mp, err))
      return ngap_fail(NGAP_ERR_INVALID, err);
    if (o.algorithm == NGAP_ALGO_BLOCKING)
      return ngap_fail(NGAP_ERR_INVALID, "blockinggroups has no batched form: use ngap_run");
    if (!ring_of(o))
      return ngap_fail(NGAP_ERR_INVALID, "ring_capacity must be a power of two in [64, 2048]");
    KParams P = base_params(eng, mp, o);
    P.ring_cap = ring_of(o);
    P.input = d_input;
    set_chunk_len(P, (uint32_t)chunk_len);
    P.num_seg = num_seg;
    // the schedule: all-group windows (depth >= 2) or one group per work item,
    // windows as ngap_run's, on a grid sized to the job
    const uint32_t G = (uint32_t)eng->img.num_groups;
    P.gen_cross = mp.memo_depth >= 2 && o.cross_groups != 0;
    const uint64_t total = (uint64_t)num_seg * chunk_len;
    const uint64_t work = total * (P.gen_cross ? 1 : G);
    P.scan = P.gen_cross && scan_image(eng, mp, total);
    P.even = P.gen_cross;
    P.load_last = (uint32_t)(total - std::min<uint64_t>(total, 8));
    const int kind = P.scan ? 6 : 4;  // of generated work items
    uint32_t blocks = 0;
    int rc = persistent_blocks(eng, o.persistent_blocks, &blocks, P.ring_cap, kind);
    if (rc) return rc;
    // a grid as asked for has to leave each wave a worklist
    if (o.persistent_blocks &&
        kScratchSpill / ((uint64_t)o.persistent_blocks * P.waves_per_block * 8) < kWave)
      return ngap_fail(NGAP_ERR_INVALID, "grid too large for the scratch array's worklists");
    uint32_t fewer = blocks;  // the grid that gives each wave a larger worklist
    if (!o.persistent_blocks) {
      fewer = job_blocks(blocks, P.waves_per_block, work, kSpillPositions);
      blocks = eng->ctx.scratch_few ? fewer : job_blocks(blocks, P.waves_per_block, work);
    }
    const uint64_t waves = (uint64_t)blocks * P.waves_per_block;
    uint32_t win = o.window;
    if (!win && P.gen_cross) {
      win = cross_window(work, waves);
      while (win < 65536 && (total / win + num_seg) * 4 > kScratchFlags) win *= 2;
    } else if (!win) {
      win = 256;
      while (win < 65536 && (double)win * 1.41421356 < (double)work / (2.0 * waves)) win *= 2;
    }
    if (win > chunk_len) win = (uint32_t)chunk_len;
    P.gen_window = win;
    const uint64_t per_chunk = (chunk_len + win - 1) / win;
    const uint64_t T = per_chunk * num_seg * (P.gen_cross ? 1 : G);
    if (T * 4 > kScratchFlags)
      return ngap_fail(NGAP_ERR_INVALID, "too many work items for the scratch array (" +
                                             std::to_string(T) + " > " +
                                             std::to_string(kScratchFlags / 4) +
                                             "): use a larger window");
    P.tasks = nullptr;
    P.num_tasks = (uint32_t)T;
    P.task_items = nullptr;
    unsigned char *base = static_cast<unsigned char *>(eng->scratch);
    unsigned long long *counters = reinterpret_cast<unsigned long long *>(base);
    P.report_count = counters + 0;
    P.items = counters + kItemsWord;
    P.overflow_count = reinterpret_cast<uint32_t *>(counters + 3);
    P.task_head = reinterpret_cast<uint32_t *>(counters + 16);
    P.overflow = reinterpret_cast<uint32_t *>(base + kScratchCounters);
    P.spill = reinterpret_cast<uint64_t *>(base + kScratchCounters + kScratchFlags);
    P.reports = d_reports;
    P.report_cap = report_cap;
    RunCtx &ctx = eng->ctx;
    float ms = 0, all_ms = 0;
    unsigned long long cnt[4];
    for (;;) {
      // spill areas: what the scratch array holds for this grid, at most the
      // requested capacity
      const uint64_t fit = kScratchSpill / ((uint64_t)blocks * P.waves_per_block * 8);
      if (fit < kWave)
        return ngap_fail(NGAP_ERR_INVALID, "grid too large for the scratch array's worklists");
      P.spill_cap = (uint32_t)std::min<uint64_t>(o.spill_capacity ? o.spill_capacity : fit, fit);
      HIP_TRY(launch_reset(ctx.stream, P.report_count, P.items, P.task_head, P.overflow,
                           P.num_tasks, P.overflow_count, 0, nullptr));
      HIP_TRY(hipEventRecord(ctx.ev0, ctx.stream));
      HIP_TRY(launch_batched(ctx.stream, P, blocks, batched_lds(P.ring_cap, kind, G)));
      HIP_TRY(hipEventRecord(ctx.ev1, ctx.stream));
      HIP_TRY(hipMemcpyAsync(ctx.host_cnt, counters, kCounterBytes, hipMemcpyDeviceToHost,
                             ctx.stream));
      HIP_TRY(hipStreamSynchronize(ctx.stream));
      HIP_TRY(hipEventElapsedTime(&ms, ctx.ev0, ctx.ev1));
      all_ms += ms;
      memcpy(cnt, ctx.host_cnt, 32);
      cnt[1] = items_sum(ctx.host_cnt);
      // what a worklist of the larger grid could not hold, the smaller grid's may
      if ((uint32_t)cnt[3] == 0 || blocks <= fewer) break;
      blocks = fewer;
      ctx.scratch_few = true;
    }
    ms = all_ms;
    if (st) {
      st->kernel_ms = ms;
      st->reports_raw = cnt[0];
      st->items = cnt[1];
      st->overflow_units = (uint32_t)cnt[3];
      st->num_units = G * num_seg;
      st->num_tasks = (uint32_t)T;
    }
    if ((uint32_t)cnt[3])
      return ngap_fail(NGAP_ERR_OVERFLOW,
                       "worklist spill capacity exceeded in " + std::to_string((uint32_t)cnt[3]) +
                           " work items (scratch worklists of " + std::to_string(P.spill_cap) +
                           " items per wave; no fallback without allocation)");
    if (cnt[0] > report_cap)
      return ngap_fail(NGAP_ERR_OVERFLOW, "report capacity exceeded: " + std::to_string(cnt[0]) +
                                              " reports > " + std::to_string(report_cap));
    return NGAP_OK;
  });
}
