// gt_bandpass_f32.hip -- the streaming bandpass for float32 frames.
#include "gt_bandpass.h"

namespace gt {
template hipError_t launch_bandpass_t<float>(int, const Batch&, const K1Params&, bool, hipStream_t);
}  // namespace gt
