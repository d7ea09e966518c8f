// The streaming top-k kernels without the large-K rank and tail, and the
// launch that picks between those and the others.
#include "stream_kernel.h"

namespace llmhip {

template hipError_t launch_stream_k<false, false>(const SampleArgs&, hipStream_t);

// bigk: some row of the launch has K > 64; refine: some row raises its
// threshold (and bigk).
hipError_t launch_stream(const SampleArgs& a, bool bigk, bool refine, hipStream_t s) {
  if (refine) return launch_stream_k<true, true>(a, s);
  return bigk ? launch_stream_k<true, false>(a, s) : launch_stream_k<false, false>(a, s);
}

}  // namespace llmhip
