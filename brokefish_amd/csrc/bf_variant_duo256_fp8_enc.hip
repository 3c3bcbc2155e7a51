// Encoder-only form of kernel variant "duo256_fp8" (e4m3, two positions per workgroup), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_duo256_fp8_enc(const KArgs& k, hipStream_t stream) { return duo::launch_duo<MODE_ENC, true>(k, stream); }
}  // namespace bf
