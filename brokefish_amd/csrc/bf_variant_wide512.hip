// Kernel variant "wide512" of the evaluator (512-wide network, two positions per workgroup), compiled as its own translation unit.
#include "bf_wide.hip.h"

namespace bf {
hipError_t launch_wide512(const KArgs& k, hipStream_t stream) { return wide::launch_wide<MODE_EVAL>(k, stream); }
}  // namespace bf
