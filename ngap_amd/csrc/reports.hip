// Sorting the reports of a run on the device: ngap_get_reports' sort by
// (offset, id), removal of repeats and change to the reference encoding
// (the reference packs and sorts them on the host, code/src/ngap/ngap.cu:
// 1899-1933, compareResult :19-30).
//
// Device reports are (offset << 32) | id, all different from ~0 (offsets stay
// below 2^32 - 2^20), so numeric order is the reference's order and ~0 marks
// an empty slot.
//  * Up to kSmallReports: a rank sort.  Every key's place is the number of
//    smaller keys, found by comparing it with all of them: n^2 comparisons,
//    but no passes and no barriers between them, so the whole chip works on
//    one launch.  Equal keys get the same place, which leaves the repeats'
//    slots empty: the second launch closes the gaps, swaps the halves and
//    writes the result straight to pinned host memory.
//  * Above: rocPRIM's radix sort and unique, in place in the report buffer
//    (reports_large.hip, a module of its own: a process's first use of rocPRIM's
//    kernels loads them, 4 ms that few reports need not wait for).
// The line between them: two ngap_get_reports calls (count, then copy) over
// 2,048 reports take 25 us, over 4,096 31, 8,192 44, 16,384 70 by rank; by radix
// (about 10 launches, the copy by hipMemcpy) over 16,385 98 to 146, 40,000 209,
// 131,072 548, 154,507 194 (the library sorts in another way from some size on),
// 1,000,000 1,520.  One 1,024-thread workgroup closes the gaps of at most 16 slots
// per thread, held in registers, which is the other reason for the line.  The
// host's std::sort, run by both calls, took 158 us over 2,522 reports, 840 over
// 13,997, 8,100 over 154,507 and 26,100 over 1,000,000.  The rank kernel is bound by its 64-bit comparisons: 14k
// keys in 59 us with a scalar load per key, 39 with one per eight.
#include <hip/hip_runtime.h>

#include "runtime.h"

namespace ngapamd {

namespace {

constexpr uint64_t kEmptySlot = ~0ull;
constexpr uint32_t kSortThreads = 1024, kSortWaves = kSortThreads / kWave;
constexpr uint32_t kKeysPerLane = kSmallReports / kSortThreads;

__device__ __forceinline__ uint64_t encode(uint64_t k) { return (k << 32) | (k >> 32); }

// slots[number of keys below keys[i]] = keys[i].  One workgroup ranks 64 keys
// (a lane each); its 16 waves each compare them with a sixteenth of all keys,
// read at wave-uniform addresses through the scalar cache.
__global__ void __launch_bounds__(kSortThreads)
    k_rank_reports(const uint64_t *__restrict__ keys, uint32_t n, uint64_t *__restrict__ slots) {
  __shared__ uint32_t part[kSortWaves][kWave];
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t i = blockIdx.x * kWave + lane;
  const uint64_t key = i < n ? keys[i] : 0;
  const uint32_t per = (n + kSortWaves - 1) / kSortWaves;
  const uint32_t end = min(n, (wave + 1) * per);
  uint32_t r = 0;
  uint32_t j = wave * per;
  const uint64_t *at = keys + j;  // constant offsets from it: one wide scalar load per 8 keys
  for (; j + 8 <= end; j += 8, at += 8) {
    uint64_t k[8];
#pragma unroll
    for (int x = 0; x < 8; x++) k[x] = at[x];
#pragma unroll
    for (int x = 0; x < 8; x++) r += k[x] < key;
  }
  for (; j < end; j++, at++) r += *at < key;
  part[wave][lane] = r;
  __syncthreads();
  if (wave == 0 && i < n) {
    uint32_t rank = 0;
#pragma unroll
    for (uint32_t w = 0; w < kSortWaves; w++) rank += part[w][lane];
    slots[rank] = key;
  }
}

// Closes the gaps (one workgroup): out[1..] = the filled slots in order,
// encoded, out[0] = their number.  The slots are left empty for the next use.
__global__ void __launch_bounds__(kSortThreads)
    k_close_gaps(uint64_t *__restrict__ slots, uint32_t n, uint64_t *__restrict__ out) {
  __shared__ uint32_t count[kSortWaves];
  const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const uint32_t base = wave * kWave * kKeysPerLane;
  uint64_t key[kKeysPerLane];
  uint32_t at[kKeysPerLane], total = 0;
#pragma unroll
  for (uint32_t k = 0; k < kKeysPerLane; k++) {
    const uint32_t i = base + k * kWave + lane;
    key[k] = i < n ? slots[i] : kEmptySlot;
  }
#pragma unroll
  for (uint32_t k = 0; k < kKeysPerLane; k++) {
    const uint64_t m = __ballot(key[k] != kEmptySlot);
    at[k] = total + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                              __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    total += __popcll(m);
  }
  if (lane == 0) count[wave] = total;
  __syncthreads();
  uint32_t before = 0;
  for (uint32_t w = 0; w < wave; w++) before += count[w];
#pragma unroll
  for (uint32_t k = 0; k < kKeysPerLane; k++) {
    if (key[k] == kEmptySlot) continue;
    out[1 + before + at[k]] = encode(key[k]);
    slots[base + k * kWave + lane] = kEmptySlot;
  }
  if (threadIdx.x == kSortThreads - 1) out[0] = before + total;
}

}  // namespace

hipError_t sort_reports_device(RunCtx &ctx, uint64_t n, uint32_t offset_bits) {
  if (n > kSmallReports) return sort_reports_large(ctx, n, 32 + offset_bits);
  hipLaunchKernelGGL(k_rank_reports, dim3(((uint32_t)n + kWave - 1) / kWave), dim3(kSortThreads),
                     0, ctx.stream, ctx.reports.as<uint64_t>(), (uint32_t)n,
                     ctx.report_slots);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_close_gaps, dim3(1), dim3(kSortThreads), 0, ctx.stream,
                     ctx.report_slots, (uint32_t)n, ctx.host_reports);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = hipStreamSynchronize(ctx.stream)) != hipSuccess) return e;
  ctx.unique_reports = ctx.host_reports[0];
  ctx.sorted_on_host = true;
  return e;
}

}  // namespace ngapamd
