// Legal-move words on the device: packed positions -> [n, 32] x u64 masks (+ in-check flags), so
// the mask the evaluator ANDs in and the expansion walks never leaves the GPU.
// Replaces env.movegen of the reference (docs/reference/spec.md:152-172; rule behaviour
// brokefish/env/torch_impl.py:77-126 pawns / en passant, :161-181 castling, :251-289 legality by
// replaying every pseudo-legal move); the CPU generator of this repository (chessgen.c, pinned by
// the published perft counts) is its checker.
//
// Four positions per wavefront, a row of sixteen lanes each: lane s of the row holds slot s of the side to
// move (its kings stand in slots 15 and 31, its colours in slots 0..15 and 16..31 by the format) and
// slot s of the other side.  The bitboards every lane needs (own pieces, the enemy's pieces by kind)
// are OR-reductions over the row.  A slider's reach along a line is two subtractions and the other
// pieces are shift patterns, so there is no loop over squares.  Legality takes two questions per lane
// instead of one replay per move:
//   * every lane asks which enemies attack the king once this lane's piece has left its square: none
//     -- the piece may go anywhere it reaches; one -- it must capture that one or step between it and
//     the king; two -- no move of it helps.  This is what replaying each of its moves would answer:
//     a piece put on a square can only take the enemy there or block a line.
//   * lanes 0..7 each try one king step, lanes 8..13 the three squares of either castling, on the
//     position after the move.
// En passant, where two pieces leave the board's lines at once, is replayed (a loop that hardly ever
// runs).  Integer work, bound by the vector ALU: one wavefront per position (its boards built on the
// scalar unit, each of some 31 moves replayed) took 119 us for 65536 positions, this 24 us, with the squares'
// diagonals, knight's and king's steps looked up (651 vector instructions a wavefront, by counter) 19 us, and with
// three-operand logic, sums for differences and pawns' squares from the king's steps (547) 17 us (1.25 TB/s of its
// bytes).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

#include "bf_args.h"
#include "bf_movegen.hip.h"

namespace {

__global__ __launch_bounds__(256) void movegen_kernel(const uint16_t* boards, const int16_t* control, int n,
                                                      uint64_t* mask, uint8_t* in_check) {
    __shared__ bf::moves::Table table;
    bf::moves::fill(table);
    const int lane = threadIdx.x & 63, slot = lane & 15;
    const int b_ = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 4);
    const bool here = b_ < n;
    const int b = here ? b_ : n - 1;                    // a row past the end repeats the last position and stores nothing
    const bool black = control[b] < 0;
    const uint64_t legal = bf::moves::of_row(boards + (size_t)b * 32, black, lane, table, [&](bool attacked) {
        if (slot == 15 && in_check && here) in_check[b] = attacked;
    });
    if (here) {
        uint64_t* const mw = mask + (size_t)b * 32;
        mw[(black ? 16 : 0) + slot] = legal;
        mw[(black ? 0 : 16) + slot] = 0;
    }
}

}  // namespace

extern "C" int bf_movegen(const uint16_t* boards, const int16_t* control, int64_t n, uint64_t* mask,
                          uint8_t* in_check, void* stream) {
    auto fail = [](int code, const char* msg) {
        bf::set_error(msg);
        return code;
    };
    if (n < 1 || n > (1ll << 28)) return fail(BF_ERR_ARGUMENT, "n must be in [1, 2^28]");
    if (!boards || !control || !mask) return fail(BF_ERR_ARGUMENT, "boards/control/mask must not be NULL");
    if (((uintptr_t)boards & 1) || ((uintptr_t)control & 1) || ((uintptr_t)mask & 7))
        return fail(BF_ERR_ARGUMENT, "boards and control must be 2-byte and mask 8-byte aligned");
    // Sixteen positions per workgroup, whatever the launch.  Workgroups of one wavefront, which spread a small one over more
    // compute units and compute the table's fields, are no faster anywhere (64 positions 4.5 us alone against 3.9, 250
    // 4.6 / 4.3, 1024 4.5 / 4.4, 4096 4.7 / 4.6, 8192 5.8 / 5.5).
    hipLaunchKernelGGL(movegen_kernel, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, (hipStream_t)stream, boards, control, (int)n, mask,
                       in_check);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        char msg[256];
        snprintf(msg, sizeof(msg), "kernel launch failed: %s", hipGetErrorString(e));
        return fail(BF_ERR_LAUNCH, msg);
    }
    return BF_OK;
}
