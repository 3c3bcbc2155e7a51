// Encoder-only form of kernel variant "ragged256_fp8" (two positions per workgroup, the last round one, e4m3), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_ragged256_fp8_enc(const KArgs& k, hipStream_t stream) { return duo::launch_ragged<MODE_ENC, true>(k, stream); }
}  // namespace bf
