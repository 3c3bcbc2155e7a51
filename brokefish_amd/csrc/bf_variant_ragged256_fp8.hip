// Kernel variant "ragged256_fp8" (two positions per workgroup, the last round one, e4m3), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_ragged256_fp8(const KArgs& k, hipStream_t stream) { return duo::launch_ragged<MODE_EVAL, true>(k, stream); }
}  // namespace bf
