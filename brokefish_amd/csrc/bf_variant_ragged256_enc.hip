// Encoder-only form of kernel variant "ragged256" (two positions per workgroup, the last round one), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_ragged256_enc(const KArgs& k, hipStream_t stream) { return duo::launch_ragged<MODE_ENC, false>(k, stream); }
}  // namespace bf
