// The streaming top-k kernels for launches with some row that raises its
// threshold as it streams.
#include "stream_kernel.h"

namespace llmhip {

template hipError_t launch_stream_k<true, true>(const SampleArgs&, hipStream_t);

}  // namespace llmhip
