// Encoder-only form of kernel variant "octo256_fp8" (eight wavefronts per position), compiled as its own translation unit.
#include "bf_board.hip.h"

namespace bf {
hipError_t launch_octo256_fp8_enc(const KArgs& k, hipStream_t stream) { return board::launch_board<256, MODE_ENC, true, true, true>(k, stream); }
}  // namespace bf
