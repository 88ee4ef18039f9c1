// A request launch's set-up and its results, one kernel each.
//
// A launch takes dozens of requests, each in a pinned host buffer of its own,
// and is bound by the host: a copy per request, a map and a work-item list
// built on the host and copied, took 50 calls of 8 us (192 requests of 1 KiB to
// 1 MiB in four launches: 2.1 to 4.3 ms after their submission, by how the runtime
// moved the copies; 1.5 now).  So the host writes 32 bytes a request and the
// device does the rest:
//  * k_gather reads the requests' bytes straight from the pinned buffers, 16
//    bytes a lane and four loads in flight, which is what the link takes (7.5 MB in
//    0.135 ms, 55 GB/s, where no other launch reads); the same kernel clears the
//    run's counters and flags, sets the map of the requests' last bytes and lists
//    the work items.
//  * k_results writes the counters and the first reports to pinned memory, where
//    retiring the launch finds them without another copy.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "runtime.h"

namespace ngapamd {

namespace {

constexpr uint32_t kThreads = 256, kUnit = 16, kUnitsPerLane = 4;

// The last of n entries whose `first` is not above x (entry 0's is 0).
template <class T>
__device__ __forceinline__ uint32_t entry_of(const T *e, uint32_t n, uint32_t x) {
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) / 2;
    if (e[mid].first <= x) lo = mid;
    else hi = mid;
  }
  return lo;
}

__global__ void __launch_bounds__(kThreads) k_gather(RequestBatch B) {
  const uint32_t at = blockIdx.x * kThreads + threadIdx.x, step = gridDim.x * kThreads;
  const uint32_t n = B.count;
  // the bytes: a wave's units lie together, 4 KiB of them
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t u0 = at / kWave * (kWave * kUnitsPerLane) + lane;
  if (u0 < B.units) {
    uint32_t r = entry_of(B.spans, n, u0);
    uint4 v[kUnitsPerLane];
    uint32_t to[kUnitsPerLane], len[kUnitsPerLane];
#pragma unroll
    for (uint32_t j = 0; j < kUnitsPerLane; j++) {
      const uint32_t u = u0 + j * kWave;
      len[j] = 0;
      if (u >= B.units) continue;
      while (r + 1 < n && B.spans[r + 1].first <= u) r++;
      const RequestSpan s = B.spans[r];
      const uint32_t o = (u - s.first) * kUnit;
      v[j] = *reinterpret_cast<const uint4 *>(s.src + o);  // the buffers are larger by far
      to[j] = s.base + o;
      len[j] = min(kUnit, s.len - o);
    }
#pragma unroll
    for (uint32_t j = 0; j < kUnitsPerLane; j++) {
      if (len[j] == kUnit) {
        __builtin_memcpy(B.input + to[j], &v[j], kUnit);  // at any alignment
      } else {
        const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
        for (uint32_t b = 0; b < kUnit; b++)
          if (b < len[j]) B.input[to[j] + b] = (uint8_t)(w[b / 4] >> (8 * (b % 4)));
      }
    }
  }
  // the run's counters, the work items' flags and the work items
  if (at == 0) {
    for (uint32_t k = 0; k < 4; k++) B.counters[k] = 0;
    for (uint32_t k = 0; k < kQueues; k++) B.task_head[k * kQueueStride] = 0;
  }
  if (at < kItemLanes) B.items[at * kItemStride] = 0;
  for (uint32_t t = at; t < B.num_tasks; t += step) {
    B.overflow[t] = 0;
    const RequestTasks q = B.order[entry_of(B.order, n, t)];
    const RequestSpan s = B.spans[q.request];
    const uint32_t a = s.base + (t - q.first) * B.window, end = s.base + s.len;
    Task T;
    T.group = s.group;
    T.cstart = s.base;
    T.cend = end;
    T.begin = a;
    T.end = min(a + B.window, end);
    T.flags = a == s.base ? kTaskSeedStart : 0u;
    B.tasks[t] = T;
  }
  // a bit per byte, set where a request ends
  for (uint32_t w = at; w < B.map_words; w += step) {
    const uint32_t lo = w * 32;
    uint32_t bits = 0;
    if (lo < B.bytes) {
      // the request that byte `lo` is in, by its base
      uint32_t x = 0, y = n;
      while (y - x > 1) {
        const uint32_t mid = (x + y) / 2;
        if (B.spans[mid].base <= lo) x = mid;
        else y = mid;
      }
      for (; x < n; x++) {
        const uint32_t last = B.spans[x].base + B.spans[x].len - 1;
        if (last - lo >= 32) break;
        bits |= 1u << (last - lo);
      }
    }
    B.map[w] = bits;
  }
}

__global__ void __launch_bounds__(kThreads)
    k_results(const unsigned long long *counters, const uint64_t *reports, uint64_t cap,
              unsigned long long *to_counters, uint64_t *to_reports) {
  const uint32_t at = blockIdx.x * kThreads + threadIdx.x;
  if (at < 4) to_counters[at] = counters[at];
  if (at < counters[0] && at < cap) to_reports[at] = reports[at];
}

}  // namespace

hipError_t launch_gather(hipStream_t s, const RequestBatch &B) {
  const uint64_t units = ((uint64_t)B.units + kUnitsPerLane - 1) / kUnitsPerLane;
  // a lane for every four units, and enough for the work items and the map
  const uint64_t want = std::max<uint64_t>(units, std::max(B.num_tasks, B.map_words / 4));
  const uint32_t blocks =
      (uint32_t)((std::max<uint64_t>(want, kItemLanes) + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(k_gather, dim3(blocks), dim3(kThreads), 0, s, B);
  return hipGetLastError();
}

hipError_t launch_results(hipStream_t s, const unsigned long long *counters,
                          const uint64_t *reports, uint64_t cap, unsigned long long *to_counters,
                          uint64_t *to_reports) {
  hipLaunchKernelGGL(k_results, dim3(kSmallReports / kThreads), dim3(kThreads), 0, s, counters,
                     reports, cap, to_counters, to_reports);
  return hipGetLastError();
}

}  // namespace ngapamd
