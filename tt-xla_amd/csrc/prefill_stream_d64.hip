// The streaming prefill kernel at head size 64.
#include "prefill_stream_kernel.h"

namespace ttpa {

int launch_stream_d64(const PrefillArgs &a, hipStream_t st) { return launch_stream_d<64>(a, st); }

}  // namespace ttpa
