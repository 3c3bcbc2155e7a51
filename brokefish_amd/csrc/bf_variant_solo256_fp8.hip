// Kernel variant "solo256_fp8" of the evaluator (e4m3, one position per workgroup of eight wavefronts), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_solo256_fp8(const KArgs& k, hipStream_t stream) { return duo::launch_duo<MODE_EVAL, true, false, 1>(k, stream); }
}  // namespace bf
