// gt_bandpass_u8.hip -- the streaming bandpass for uint8 frames.
#include "gt_bandpass.h"

namespace gt {
template hipError_t launch_bandpass_t<uint8_t>(int, const Batch&, const K1Params&, bool, hipStream_t);
}  // namespace gt
