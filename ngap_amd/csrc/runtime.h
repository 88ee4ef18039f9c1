// Host-side engine state shared by the C ABI entry points (runtime.cpp) and
// the request server (server.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <string>
#include <utility>
#include <vector>

#include <memory>

#include "../../include/ngap_amd.h"
#include "host_pool.h"
#include "kernels.h"
#include "layout.h"

void ngap_set_last_error_internal(const std::string &m) noexcept;  // errors.cpp
int ngap_fail(int code, const std::string &msg);

#define HIP_TRY(expr)                                                                 \
  do {                                                                                \
    hipError_t _e = (expr);                                                           \
    if (_e != hipSuccess)                                                             \
      return ngap_fail(_e == hipErrorOutOfMemory ? NGAP_ERR_OOM : NGAP_ERR_DEVICE,    \
                       std::string(#expr) + ": " + hipGetErrorString(_e));            \
  } while (0)

namespace ngapamd {

// Device memory for one load: the builder's temporaries and the arrays it
// builds come out of a few large chunks, by best fit, and go back to them.  What
// is given back is handed out again without waiting, so all of it is used on one
// stream.  (A load made 65 hipMalloc and 65 hipFree calls, 8.5 of its 20 ms at
// 128 automata of up to 50,000 states: each free waits for the device and unmaps.
// With a few chunks, and the uploads through the pinned blocks, it takes 5.5 ms.)
// Where memory is short it hands out allocations of their own instead (direct).
class Slab {
 public:
  Slab() = default;
  Slab(const Slab &) = delete;
  Slab &operator=(const Slab &) = delete;
  ~Slab() { clear(); }
  // the size of the first chunk, where the caller can tell what it will need
  void expect(size_t bytes) { expected_ = bytes; }
  hipError_t take(size_t bytes, void **p);
  void give(void *p);
  void clear();  // frees the chunks; nothing taken may be used any more
  // (while nothing is taken) each piece its own allocation, freed when given back
  void set_direct(bool direct) { direct_ = direct; }

 private:
  struct Piece {
    size_t chunk, at, n;
  };
  std::vector<char *> chunks_;
  std::vector<Piece> free_;  // ascending (chunk, at), neighbours joined
  std::vector<std::pair<void *, Piece>> used_;
  size_t expected_ = 0, total_ = 0;
  bool direct_ = false;
};

struct DevBuf {
  void *p = nullptr;
  size_t n = 0;
  bool owned = true;  // false: a view into another buffer (the image arena)
  Slab *slab = nullptr;  // where its memory comes from (null: hipMalloc)
  DevBuf() = default;
  explicit DevBuf(Slab &from) : slab(&from) {}
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  ~DevBuf() { release(); }
  void release();
  hipError_t reserve(size_t bytes);  // grows; contents not preserved
  template <class T>
  hipError_t upload(const std::vector<T> &v) {
    hipError_t e = reserve(v.size() * sizeof(T));
    if (e != hipSuccess) return e;
    if (!v.empty()) e = hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
    return e;
  }
  template <class T>
  T *as() const { return reinterpret_cast<T *>(p); }
};

// Pinned staging of ngap_set_input and of the groups' arrays at a load: two
// blocks, so that host threads fill one while the other's copy to the device
// runs.
struct InputStage {
  static constexpr size_t kBlock = 8u << 20;
  uint8_t *buf[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};  // the block's copy to the device
  std::unique_ptr<HostPool> pool;
  InputStage() = default;
  InputStage(const InputStage &) = delete;
  InputStage &operator=(const InputStage &) = delete;
  ~InputStage() {
    for (int i = 0; i < 2; i++) {
      if (done[i]) (void)hipEventSynchronize(done[i]);
      if (buf[i]) (void)hipHostFree(buf[i]);
      if (done[i]) (void)hipEventDestroy(done[i]);
    }
  }
  // allocates what an earlier, failed call left missing
  hipError_t init() {
    for (int i = 0; i < 2; i++) {
      if (!buf[i]) {
        const hipError_t e =
            hipHostMalloc(reinterpret_cast<void **>(&buf[i]), kBlock, hipHostMallocDefault);
        if (e != hipSuccess) {
          buf[i] = nullptr;
          return e;
        }
      }
      if (!done[i]) {
        const hipError_t e = hipEventCreateWithFlags(&done[i], hipEventDisableTiming);
        if (e != hipSuccess) {
          done[i] = nullptr;
          return e;
        }
      }
    }
    if (!pool) pool.reset(new HostPool());
    return hipSuccess;
  }
};

// One stream with its own per-run buffers and captured graph.
constexpr uint32_t kSmallReports = 16384;  // sorted by rank, above by radix (reports.hip)
struct RunCtx {
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  unsigned long long *host_cnt = nullptr;  // pinned: the run's counters after finish()
  DevBuf reports, counters, overflow, spill, tasks, task_items, fb_tasks, fb_spill;
  // root pass: pieces of the resident work items, each work item's area
  // offsets (items), the areas and the per-work-item counts
  DevBuf pieces, root_off, root_items, root_count;
  uint32_t num_pieces = 0;
  // a run whose waves had less than the largest default worklists overflowed:
  // later runs of its kind do not try that again (batched; plain units on four
  // waves; ngap_run_noalloc on the smaller grid)
  bool spill_most = false, plain_few = false, scratch_few = false;
  uint32_t root_factor = 0;     // items per position the resident areas were sized for
  uint32_t root_boost = 1;      // doubles (up to 64x) after a root area overflowed,
  uint64_t root_gen = 0;        // for this engine generation (groups and input)
  uint64_t report_cap = 0, last_count = 0;
  // the last run's reports once ngap_get_reports sorted them (until the next
  // launch): unique_reports of them, encoded, in host_reports[1..] (pinned) or
  // in `reports`
  bool sorted = false, sorted_on_host = false;
  uint64_t unique_reports = 0;
  uint64_t *host_reports = nullptr;  // kSmallReports + 1 words behind host_cnt
  uint64_t *report_slots = nullptr;  // the rank sort's, behind the counters; ~0 = empty
  DevBuf sort_area;                  // the radix sort's
  bool last_report_off = false, have_run = false;
  bool tasks_resident = false;  // `tasks` holds last_tasks
  bool last_traces = false;     // the last run recorded items per work item
  uint64_t resident_sched = 0;  // schedule id of last_tasks (0 = unknown)
  std::vector<Task> last_tasks;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  std::vector<unsigned char> gkey;
  RunCtx() = default;
  RunCtx(const RunCtx &) = delete;
  ~RunCtx();
  int init();
  void drop_graph();
  // Whether the counters and the first n words of `overflow` are known to be
  // zero: the last finish() on them left them so.  Each launch takes it back.
  bool counters_zero = false;
  const void *zero_flags = nullptr;
  size_t zero_cap = 0;
  uint32_t zero_n = 0;
  // Clears P's counters and n flags on the stream, where they are not zero yet.
  int begin(const KParams &P, uint32_t n, bool keep_reports);
  // Ends a timed launch begun with ev0: records ev1 (unless the launch
  // recorded it), queues k_finish (the run counters into host_cnt) behind
  // it and waits for the stream once.  *ms = ev0..ev1; cnt = reports, items
  // (the lanes summed), -, overflowed units.
  int finish(float *ms, unsigned long long cnt[4], bool record_end);
};

struct Mapping {
  int memo_depth;
  int priv_limit;
  int root_batch;  // positions per root step of per-group work
};

bool map_algorithm(int algorithm, int depth_req, int loaded_depth, Mapping &m, std::string &err);

// Sorts ctx's last n reports (offsets below 2^offset_bits) on the device and
// encodes them (reports.hip): into ctx.host_reports[1..] up to kSmallReports,
// else in place in ctx.reports.  Sets ctx.unique_reports and
// ctx.sorted_on_host.
hipError_t sort_reports_device(RunCtx &ctx, uint64_t n, uint32_t offset_bits);
hipError_t sort_reports_large(RunCtx &ctx, uint64_t n, uint32_t bits);

// What the device needs to set up a request launch (requests.hip): the requests
// in the order of their bytes in the input, each with its first 16-byte unit, and
// in the order of the work items, longest first, each with its first work item.
struct RequestSpan {
  const uint8_t *src;  // pinned, 16-byte aligned, readable to a multiple of 16
  uint32_t base, len, group, first;
};
struct RequestTasks {
  uint32_t first, request;
};
struct RequestBatch {
  const RequestSpan *spans;
  const RequestTasks *order;
  uint32_t count, units, bytes, window, num_tasks, map_words;
  uint8_t *input;
  uint32_t *map;
  Task *tasks;
  uint32_t *overflow, *task_head;
  unsigned long long *counters, *items;
};
hipError_t launch_gather(hipStream_t s, const RequestBatch &B);
// counters[0..3] and the first min(count, cap, kSmallReports) reports, to pinned memory
hipError_t launch_results(hipStream_t s, const unsigned long long *counters,
                          const uint64_t *reports, uint64_t cap, unsigned long long *to_counters,
                          uint64_t *to_reports);

// The request servers of an engine (ngap_server_create adds, ngap_server_destroy
// removes; shared, since either may be destroyed first).
struct ServerList {
  std::vector<ngap_server *> all;
};
// Retires every launch in flight on the engine's servers, re-runs of overflowed
// ones included.  Their kernels hold raw pointers into the image, whose memory
// the next load reuses, so a load begins with this.
int settle_servers(ngap_engine *eng);

// Kernel launchers (kernels.hip).  launch_reset clears the run's counters
// and n per-work-item flags (and root counts, when given); launch_roots runs
// the root pass (k_roots) over P.pieces.
hipError_t launch_reset(hipStream_t s, unsigned long long *rc, unsigned long long *items,
                        uint32_t *head, uint32_t *ovf, uint32_t n, uint32_t *ovf_count,
                        int keep_reports, unsigned long long *root_count);
hipError_t launch_finish(hipStream_t s, unsigned long long *counters, unsigned long long *to);
hipError_t launch_plain(hipStream_t s, const KParams &P, uint32_t units, uint32_t lds);
hipError_t launch_blocking(hipStream_t s, const KParams &P, uint32_t units, uint32_t lds);
hipError_t launch_roots(hipStream_t s, const KParams &P, uint32_t lds);
hipError_t launch_batched(hipStream_t s, const KParams &P, uint32_t blocks, uint32_t lds);
hipError_t batched_occupancy(int *blocks_per_cu, uint32_t lds, int kind);  // kind: batched_kind()
hipError_t set_lds_limit(uint32_t lds);  // of every kernel with dynamic LDS

}  // namespace ngapamd

struct ngap_engine {
  int device = 0;
  int num_cus = 0;
  // blocks per CU by (log2(ring), batched kernel kind) for the loaded groups,
  // 0 = not queried
  int batched_per_cu[12 * ngapamd::kBatchedKinds] = {0};
  ngapamd::Image img;
  bool loaded = false;
  std::shared_ptr<ngapamd::ServerList> servers = std::make_shared<ngapamd::ServerList>();
  ngapamd::Slab build_slab;  // the device builder's memory while a load runs
  ngapamd::DevBuf d_meta, d_succ4, d_cls, d_sod, d_mask1;
  ngapamd::DevBuf d_beg[ngapamd::kMaxMemoDepth], d_nrep[ngapamd::kMaxMemoDepth],
      d_list[ngapamd::kMaxMemoDepth], d_filt[ngapamd::kMaxMemoDepth],
      d_sel[ngapamd::kMaxMemoDepth];
  ngapamd::DevBuf d_xr1, d_xe1, d_xmask1, d_xr2, d_xe2, d_xsod, d_xs3, d_xp3, d_xf3, d_xb3,
      d_x2rep;
  std::array<ngapamd::DevBuf *, 31> image_arrays() {
    return {&d_succ4, &d_cls, &d_xs3, &d_xp3, &d_xf3, &d_xb3, &d_list[0], &d_list[1],
            &d_list[2], &d_filt[0], &d_filt[1], &d_filt[2], &d_sel[0], &d_sel[1], &d_sel[2],
            &d_beg[0], &d_beg[1], &d_beg[2], &d_nrep[0], &d_nrep[1], &d_nrep[2], &d_xr1,
            &d_xe1, &d_xmask1, &d_xr2, &d_xe2, &d_xsod, &d_x2rep, &d_meta, &d_sod, &d_mask1};
  }
  // one allocation holding every image array above (they are views into it)
  ngapamd::DevBuf d_arena;
  ngapamd::DevBuf d_input;
  ngapamd::InputStage stage;    // pinned staging of ngap_set_input and of loads
  uint64_t chunk_len = 0;
  uint32_t num_seg = 0;
  bool have_input = false;
  double byte_freq[256] = {0};  // input byte histogram (normalised)
  ngapamd::RunCtx ctx;          // the context ngap_run uses
  // last schedule built by ngap_run, reused while its inputs are unchanged
  struct SchedCache {
    uint64_t id = 0;            // 0 = empty; ids are never reused
    uint64_t generation = 0;    // engine generation it was built for
    int kind = -1;              // 0 host work items, 1 all-group, 2 per-group
    uint32_t window = 0, waves = 0;
    int is_dup = 0, memo_depth = 0;
    std::vector<ngap_task> host;
    std::vector<ngapamd::Task> tasks;
  } sched;
  uint64_t generation = 1;      // bumped by ngap_load_groups / ngap_set_input
  void *scratch = nullptr;      // device address of this device's scratch array
                                // (ngap_run_noalloc)
  ngapamd::ImageSizes img_sizes;  // bytes of each device image array
  bool built_on_device = false;   // the last ngap_load_groups built on the device
  double build_ms = 0;            // its wall time
};

namespace ngapamd {
KParams base_params(const ngap_engine *eng, const Mapping &mp, const ngap_run_opts &o);
void attach_ctx(KParams &P, RunCtx &ctx);
int engine_kind(const ngap_run_opts &o, bool scan);
// Whether all-group work items of this engine's runs take k_scan: memo depth
// 3, no depth-1 or depth-2 reports in the image, records and classes below
// 4 GiB each, and an input that holds an 8-byte load.  It is the faster one
// wherever it can run: 0.120 ms against the general kernel's 0.161 (400,000 states,
// 16 MiB), 0.191 / 0.194 (1,024 automata, 8 MiB), 1.11 / 1.13 (64 MiB), 0.100 / 0.114
// (short words in text), 0.026 / 0.030 (DNA literals, 1 MiB).
bool scan_image(const ngap_engine *eng, const Mapping &mp, uint64_t input_len);
// Persistent grid of the batched kernel `kind` (batched_occupancy) for ring.
int persistent_blocks(const ngap_engine *eng, uint32_t requested, uint32_t *blocks,
                      uint32_t ring = kRing, int kind = 1);
// The default persistent grid for a job of `work` positions (summed over the
// groups each work item scans): the full grid, or fewer workgroups when that
// would leave a wave fewer than kMinWavePositions positions, one search step of
// k_scan (DNA literals: 1 MiB 0.026 ms on the full grid, 0.031 on 384 workgroups;
// 64 KiB 0.017 on 128, 0.019 on 64).
constexpr uint64_t kMinWavePositions = 128;
uint32_t cross_window(uint64_t positions, uint64_t waves);
uint32_t job_blocks(uint32_t full_blocks, uint32_t waves_per_block, uint64_t work,
                    uint64_t per_wave = kMinWavePositions);
// Positions for which a wave's default worklist (64K items) was sized: a job on
// more waves than one per so many has smaller ones, so that the grids of small
// jobs cost no more memory (1 MiB of DNA, the first run of an engine 0.69 ms with
// 2 GiB to allocate, 0.39 so).
constexpr uint64_t kSpillPositions = 640;
uint32_t ring_of(const ngap_run_opts &o);
// Runs tasks on ctx (batched kernel), with the overflow fallback of o.
int run_tasks(ngap_engine *eng, RunCtx &ctx, KParams P, const std::vector<Task> &tasks,
              uint64_t sched_id,
              const ngap_run_opts &o, ngap_run_stats *st);
// Device reports of ctx's last run, sorted and unique (device encoding).
int sorted_reports(RunCtx &ctx, std::vector<uint64_t> &out);
// Builds the image of the groups on the device into eng's image buffers
// (build.hip): the arrays build_image makes, byte for byte.  img gets the
// parts the host reads (group metadata, root masks, counts), sz the arrays'
// sizes.  Returns a status; err holds the message.
int build_image_device(ngap_engine *eng, const HostGroup *groups, int32_t num_groups,
                       int32_t depth, hipStream_t s, Image &img, ImageSizes &sz,
                       std::string &err);
// With `device` current: the device address of that device's copy of the
// scratch array of ngap_run_noalloc (looked up once per device).
int noalloc_attach(int device, void **out);
}  // namespace ngapamd
