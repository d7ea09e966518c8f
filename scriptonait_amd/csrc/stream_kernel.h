// The streaming top-k kernel (stream_row.h) and its launch, templated on
// BIGK (some row has K > 64) and REFINE (some row raises its threshold): each
// instantiation is compiled in a file of its own (stream_topk.hip,
// stream_topk_bigk.hip, stream_topk_refine.hip).
#pragma once
#include <algorithm>

#include "stream_row.h"

namespace llmhip {

template <bool TAIL, bool FULL, bool BIGK, bool REFINE>
__global__ __launch_bounds__(kBlock) void sample_stream_kernel(SampleArgs a) {
  __shared__ StreamKernelLds L;
  stream_rows<TAIL, FULL, BIGK, REFINE>(a, L);
}

// One persistent workgroup per CU (at most one per row).
template <bool BIGK, bool REFINE>
hipError_t launch_stream_k(const SampleArgs& a0, hipStream_t s) {
  SampleArgs a = a0;
  a.launch_rows = launch_grid(a);
  if (a.launch_rows == 0) return hipSuccess;
  const uint32_t grid = std::min(a.launch_rows, std::max(a.cus, 1u));
  const bool full = a.allowed || a.allowed_bits || a.ring_cap;
  // A row's last float4 may pass V where it then still lies in the row's
  // 16-byte aligned stride; elsewhere it could pass the end of the buffer.
  const bool tail = a.V % 4u != 0u && (reinterpret_cast<uintptr_t>(a.logits) % 16u != 0u || a.ld % 4u != 0u);
  if (tail && full) {
    hipLaunchKernelGGL((sample_stream_kernel<true, true, BIGK, REFINE>), dim3(grid), dim3(kBlock), 0, s, a);
  } else if (tail) {
    hipLaunchKernelGGL((sample_stream_kernel<true, false, BIGK, REFINE>), dim3(grid), dim3(kBlock), 0, s, a);
  } else if (full) {
    hipLaunchKernelGGL((sample_stream_kernel<false, true, BIGK, REFINE>), dim3(grid), dim3(kBlock), 0, s, a);
  } else {
    hipLaunchKernelGGL((sample_stream_kernel<false, false, BIGK, REFINE>), dim3(grid), dim3(kBlock), 0, s, a);
  }
  return hipGetLastError();
}

extern template hipError_t launch_stream_k<false, false>(const SampleArgs&, hipStream_t);
extern template hipError_t launch_stream_k<true, false>(const SampleArgs&, hipStream_t);
extern template hipError_t launch_stream_k<true, true>(const SampleArgs&, hipStream_t);

}  // namespace llmhip
