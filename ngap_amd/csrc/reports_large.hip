// More than kSmallReports reports sorted on the device (reports.hip has the others
// and the line between them).
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_select.hpp>

#include <algorithm>

#include "runtime.h"

namespace ngapamd {

namespace {

__global__ void k_encode(uint64_t *keys, const uint64_t *count) {
  const uint64_t n = *count;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    keys[i] = (keys[i] << 32) | (keys[i] >> 32);
}

}  // namespace

// The radix path: reports[0, n) -> sorted, unique, encoded in place.
// hipErrorOutOfMemory when its work area cannot be allocated.
hipError_t sort_reports_large(RunCtx &ctx, uint64_t n, uint32_t bits) {
  uint64_t *keys = ctx.reports.as<uint64_t>();
  size_t sort_bytes = 0, uniq_bytes = 0;
  hipError_t e = rocprim::radix_sort_keys(nullptr, sort_bytes, keys, keys, n, 0, bits, ctx.stream);
  if (e != hipSuccess) return e;
  e = rocprim::unique(nullptr, uniq_bytes, keys, keys, keys, n, rocprim::equal_to<uint64_t>(),
                      ctx.stream);
  if (e != hipSuccess) return e;
  const size_t tmp = (std::max(sort_bytes, uniq_bytes) + 255) / 256 * 256;
  if ((e = ctx.sort_area.reserve(tmp + n * 8 + 8)) != hipSuccess) return e;
  uint64_t *sorted = reinterpret_cast<uint64_t *>(ctx.sort_area.as<char>() + tmp);
  uint64_t *kept = sorted + n;
  e = rocprim::radix_sort_keys(ctx.sort_area.p, sort_bytes, keys, sorted, n, 0, bits, ctx.stream);
  if (e != hipSuccess) return e;
  e = rocprim::unique(ctx.sort_area.p, uniq_bytes, sorted, keys, kept, n,
                      rocprim::equal_to<uint64_t>(), ctx.stream);
  if (e != hipSuccess) return e;
  const uint32_t blocks = (uint32_t)std::min<uint64_t>((n + 255) / 256, 2048);
  hipLaunchKernelGGL(k_encode, dim3(blocks), dim3(256), 0, ctx.stream, keys, kept);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = hipMemcpyAsync(ctx.host_reports, kept, 8, hipMemcpyDeviceToHost, ctx.stream)) !=
      hipSuccess)
    return e;
  if ((e = hipStreamSynchronize(ctx.stream)) == hipSuccess)
    ctx.unique_reports = ctx.host_reports[0];
  return e;
}

}  // namespace ngapamd
