// The streaming prefill kernel at head size 256.
#include "prefill_stream_kernel.h"

namespace ttpa {

int launch_stream_d256(const PrefillArgs &a, hipStream_t st) { return launch_stream_d<256>(a, st); }

}  // namespace ttpa
