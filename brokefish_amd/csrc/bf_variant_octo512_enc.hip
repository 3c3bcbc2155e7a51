// Encoder-only form of kernel variant "octo512" (eight wavefronts per position), compiled as its own translation unit.
#include "bf_board.hip.h"

namespace bf {
hipError_t launch_octo512_enc(const KArgs& k, hipStream_t stream) { return board::launch_board<512, MODE_ENC, true, false, true>(k, stream); }
}  // namespace bf
