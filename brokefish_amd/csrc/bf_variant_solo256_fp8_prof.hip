// Kernel variant "solo256_fp8_prof" of the evaluator (e4m3, one position per workgroup of eight wavefronts), compiled as its own translation unit.
#include "bf_duo.hip.h"

namespace bf {
hipError_t launch_solo256_fp8_prof(const KArgs& k, hipStream_t stream) { return duo::launch_duo<MODE_EVAL, true, true, 1>(k, stream); }
}  // namespace bf
