// Encoder-only form of kernel variant "wide512" (512-wide network, two positions per workgroup), compiled as its own translation unit.
#include "bf_wide.hip.h"

namespace bf {
hipError_t launch_wide512_enc(const KArgs& k, hipStream_t stream) { return wide::launch_wide<MODE_ENC>(k, stream); }
}  // namespace bf
