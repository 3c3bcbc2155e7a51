// Encoder-only form of kernel variant "twin256_fp8" (two workgroups per compute unit), compiled as its own translation unit.
#include "bf_board.hip.h"

namespace bf {
hipError_t launch_twin256_fp8_enc(const KArgs& k, hipStream_t stream) { return board::launch_board<256, MODE_ENC, true, true>(k, stream); }
}  // namespace bf
