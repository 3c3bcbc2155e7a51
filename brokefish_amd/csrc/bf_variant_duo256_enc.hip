// Encoder-only form of kernel variant "duo256" (two positions per workgroup), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_duo256_enc(const KArgs& k, hipStream_t stream) { return duo::launch_duo<MODE_ENC, false>(k, stream); }
}  // namespace bf
