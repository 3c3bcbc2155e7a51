// Encoder-only form of kernel variant "solo256" (one position per workgroup of the two-position kernel), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_solo256_enc(const KArgs& k, hipStream_t stream) { return duo::launch_duo<MODE_ENC, false, false, 1>(k, stream); }
}  // namespace bf
