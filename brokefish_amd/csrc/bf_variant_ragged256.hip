// Kernel variant "ragged256" (two positions per workgroup, the last round one), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_ragged256(const KArgs& k, hipStream_t stream) { return duo::launch_ragged<MODE_EVAL, false>(k, stream); }
}  // namespace bf
