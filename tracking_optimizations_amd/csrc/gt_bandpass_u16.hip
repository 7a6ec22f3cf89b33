// gt_bandpass_u16.hip -- the streaming bandpass for uint16 frames.
#include "gt_bandpass.h"

namespace gt {
template hipError_t launch_bandpass_t<uint16_t>(int, const Batch&, const K1Params&, bool, hipStream_t);
}  // namespace gt
