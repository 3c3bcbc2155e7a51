// The evaluator with a TEAM of workgroups per position: the form for launches that leave most of the chip idle.
//
// A position's latency on one compute unit is bound by what that unit has to do alone: its weights cross the
// unit's 64 bytes/clock fill path (786 KB, 12.3 k clocks of a 36 k clock layer at width 256; 3.1 MB, 49 k of
// 110 k at width 512), and all heads and tiles pass through four SIMDs.  Here NWG = d_ff / 256 workgroups of eight
// wavefronts (4 at width 256, 8 at width 512), one per compute unit and all behind the same L2, share one position:
//   - the residual stream is held by every member (each wavefront 1 or 2 tiles of the width in registers), so both
//     LayerNorms, the quantisers and the output projection are computed by every member without asking another;
//   - member m has two attention heads: six wavefronts compute their Q, K and V tiles, four the attention (a
//     head's queries split in two, v_mfma_f32_16x16x4f32: the same fused-multiply-add chain in a quarter of the
//     clocks of the 32x32x2 form's tile); the heads' outputs go to everybody (exchange A);
//   - member m computes the 256 hidden channels of k-chunk m, which are one quantiser group of their own, and
//     that chunk's part of the second matmul for the whole width; the int32 (e4m3: fp32) partial accumulators
//     and the chunk's scales go to everybody (exchange B), who sums them in chunk order.
// So a layer has two exchanges (five members and more: B in two steps, each member summing the accumulators of its two
// tiles and giving the sums to all, which is a fifth of the bytes at width 512), its weights are read once per team
// except the output projection's, and a wavefront has one tile (width 512: two) in a matmul.  Measured, one position:
// 120 -> 73.8 us, e4m3 155 -> 88.7, width 512 with 16 layers 738 -> 255; 64 positions 120 -> 78.7, e4m3 155 -> 93.3; 32 of the
// wide network 738 -> 314.  The arithmetic is that of the other kernels, operation for operation: the results are
// bit-identical to theirs.
//
// Rows and tiles.  For everything per row (LayerNorm, quantisers, residual sums) a wavefront owns the rows of four
// tokens, a lane a 16-value chain of one of them, so a row's sums and maxima are a few cross-lane instructions.  With
// the accumulator layout's split (a wavefront a tile, all tokens), as the other kernels have it, each of these was an
// exchange through LDS: thirteen barriers a layer instead of seven, 90 us instead of 84.  The matmuls take the
// quantised rows from LDS; their results come back as rows through LDS (output projection) or on the way through
// the L2, where pieces are laid out so that four tokens, 64 bytes, stay together on either side.
//
// What bounds it now: a layer is some 20 k clocks at width 256, of which the waits for other members are 1.5 k; the unit's
// path to the L2 moves 370 KB in it (5.8 k clocks, most of it under something else), two LayerNorms, three
// quantisers and the epilogues are some 7 k of vector work, attention 2.8 k.  Outside the layers: 7.6 k to the first one (two
// loads that depend on each other; 8.5 k with every wavefront asking for the rows that all tokens share), 6.9 k of final norm and head
// chain (8.3 k while the chain waited for its operands out of LDS at every step), 3 k for the best move: together 75.5 -> 74.5 us, 64
// positions 81.1 -> 79.9, 20 of the wide network 300 -> 291.  (Lines of the first layer's weights and of the head tiles
// asked for ahead: 75.7.  The output projection's weights moved out of LayerNorm 1, into the QKV phase or the attention: 76.7 to 81.9.)
// The path takes a 16-byte load of 64 lanes in 16 clocks and a wavefront stops at the load that finds it busy, so where the
// loads stand matters as much as how many they are (one position, 82.3 us before):
//   - a layer's parameters, asked for right before the Q, K, V products, made those wait for them (all loads return in order);
//     the four wavefronts without attention ask for the next layer's in that time: 81.5, width 512 273 -> 265;
//   - weights between the vector instructions of the LayerNorms and the softmax instead of all at once: 78.7 (and, once the ends were shorter,
//     six instructions apart in LayerNorm 1 and fifteen in 2, not five and ten: 74.7 -> 73.8, 64 positions 79.6 -> 78.7, e4m3 90.2 -> 88.7);
//   - a member's own piece of exchange B through LDS (96 KB instead of 128), each copy of the sum in the order of the loads: 76.4.
//
// An exchange: a wavefront stores its piece, waits until the L2 has it (vmcnt), and stores a flag; the wavefronts that
// need the piece poll the flags past their L1 (sc1) and then load the piece past it (polling tags inside the data
// itself was slower: every poll is 16 KiB).  Members sit behind one L2 because workgroups go to the XCDs in turn
// (blockIdx % 8; bf_team_workspace_bytes looks at the device before the form is used).  Flags count layers, modulo 2^32, over all
// launches of a workspace (each member keeps the count), so nothing is cleared between launches.  Waiting is
// bounded: a wavefront that has waited some seconds gives up.  It publishes nothing any more, so that everybody who needs
// its pieces gives up too; its member's outputs become NaN, the best move -1, and a word in host memory tells the library,
// which reports it with the next call (BF_ERR_TEAM).
// Members of a team are consecutive workgroups of their XCD and are dispatched in order, so at most NWG - 1
// workgroups of a launch per XCD ever wait for a unit to come free.  With 32 units per XCD that allows ten launches at a
// time on a device, all processes together (width 512: four); were there more, incomplete teams could hold every unit
// of an XCD and wait for one another until they give up.  A process stays below that by itself with HIP's four
// hardware queues; with more than the bound allows (GPU_MAX_HW_QUEUES) the form is not used.
//
// One set of exchange buffers per team is enough: a member writes A, B or C of layer l + 1 only after barriers that
// follow all its wavefronts' loads of the last exchange of layer l from all members, and every wavefront loads A of a
// layer before it stores its B.
//
// LDS map: [xch: 8 waves x 64 floats] [act: the quantised rows of the width] [hid: the quantised chunk] [tok: the
// activation scales of act's rows] [par: a layer's side parameters, twice] [ex: Q, K, V of two heads; the output
// projection's tiles; the normalised stream (fp32) of the heads].
#pragma once

#include "bf_board.hip.h"

typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

namespace bf {
namespace team {

using board::chunk_sum;
using board::dma;
using board::frag_mma;
using board::lds;
using board::lds_barrier;
using board::wait_vm;

template <int DM>
struct Cfg : Layout<DM> {
    typedef Layout<DM> L;
    static constexpr int NWG = L::KCF, NW = 8;      // members of a team; wavefronts of a member
    static constexpr int TWW = L::NT / NW;          // tiles of a matmul over the width a wavefront computes
    static constexpr int NP = TWW;                  // tiles of a row a lane holds, of the four rows a wavefront owns
    static_assert(L::NT / NWG == 2, "two heads per member");
    // side parameters of a quarter in LDS: part A, the head of part B, this member's row of 128 * sum(w), its step of the hidden biases
    static constexpr int P_B = L::A_FLOATS, P_WSUM = P_B + L::B_LDS_FLOATS, P_BFF1 = P_WSUM + L::CW, P_FLOATS = P_BFF1 + 128;
    static constexpr int XCH_OFF = 0;
    static constexpr int ACT_OFF = XCH_OFF + NW * 64 * 4;
    static constexpr int HID_OFF = ACT_OFF + L::NT * FRAG;
    static constexpr int TOK_OFF = HID_OFF + 8 * FRAG;
    static constexpr int PAR_OFF = TOK_OFF + FRAG;
    static constexpr int PAR_BYTES = 4 * P_FLOATS * 4;
    static constexpr int EX_OFF = PAR_OFF + 2 * PAR_BYTES;
    static constexpr int EX_TILE = 4 * FRAG + 64;   // a tile in accumulator layout; the padding spreads the tiles of a row over the banks
    static constexpr int EX_BYTES = L::NT * EX_TILE > 24 * FRAG ? L::NT * EX_TILE : 24 * FRAG;
    static constexpr int USED_BYTES = EX_OFF + EX_BYTES;
    // more than half a compute unit's LDS: never two workgroups on one unit while another is empty
    static constexpr int LDS_BYTES = USED_BYTES < 81 * 1024 ? 81 * 1024 : USED_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
    // a team's part of the workspace, bytes.  A stream-shaped piece is [owner wave][quad 4][NP][64 lanes] 16 bytes.
    static constexpr int FLAG_A = 64, FLAG_B = 128;           // dwords: first flag of exchange A [query half][tile], of exchange B [member][wave]
    static constexpr int ROWS = L::NT * 4 * FRAG;             // a stream-shaped piece; an owner wave's part; a quad of that
    static constexpr int ROWS_W = ROWS / NW, ROWS_Q = ROWS_W / 4;
    // more than four members: exchange B in two steps, each member sums the accumulators of two tiles and gives the sums to all
    static constexpr bool TWO_STEPS = NWG > 4;
    static constexpr int WS_A = BF_TEAM_FLAG_BYTES, WS_B = WS_A + ROWS, WS_S = WS_B + NWG * ROWS;   // [member]: accumulators; scales [member][token]
    static constexpr int FLAG_C = FLAG_B + NWG * NW, FLAG_H = FLAG_C + NWG * NW, WS_H = 3072;   // heads: [policy job]; its best move, 16 bytes
    static constexpr int WS_C = WS_S + NWG * T * 4;   // the second step: [member][wave]; stream-shaped
    static constexpr int WS_BYTES = (WS_C + (TWO_STEPS ? ROWS : 0) + 4095) / 4096 * 4096;
    static_assert(NWG <= FLAG_A && FLAG_A + 2 * L::NT <= FLAG_B && (FLAG_H + 8) * 4 <= WS_H && WS_H + 8 * 16 <= WS_A, "flags");
    static_assert(!TWO_STEPS || NWG * TWW == L::NT, "a member's tiles are those of one wavefront");
    // Who waits for whom in exchange B.  A wavefront's flag stands for what that wavefront itself stored and for nothing else, so a
    // reader may load only what was stored by a wavefront whose flag it waits for (tests/test_team_exchange.py goes through all pairs).
    // In one step it waits for all wavefronts; in two, member m loads what wavefront m of every member stored, and the scales,
    // which a member's wavefront 0 stores.
    static constexpr int FLAGS_B = TWO_STEPS ? 2 * NWG : NWG * NW;
    static constexpr int flag_b(int member, int wave) { return FLAG_B + member * NW + wave; }
    static constexpr int awaited_b(int reader, int i) { return TWO_STEPS ? flag_b(i % NWG, i < NWG ? reader : 0) : flag_b(0, i); }   // the i-th of FLAGS_B
    static constexpr int scales_b(int member) { return WS_S + member * T * 4; }
    static constexpr int piece_b(int member, int tile, int quad) { return WS_B + member * ROWS + (tile * 4 + quad) * FRAG; }   // in two steps
    static constexpr int tile_b(int member, int wave) { return TWW * member + (wave >> 2); }   // the tile whose accumulators a wavefront sums, in two steps
};

// Tags count modulo 2^32 (2^31 layers are some six hours of launches in a row).  A flag of the exchanges is raised in every layer,
// so it lags by one launch at most; those of the heads are raised in launches with a best move only and may lag by any number.
struct Reached { __host__ __device__ constexpr bool operator()(unsigned flag, unsigned tag) const { return (int)(flag - tag) >= 0; } };
struct Equal { __host__ __device__ constexpr bool operator()(unsigned flag, unsigned tag) const { return flag == tag; } };

// Whether launches on `queues` hardware queues at a time, teams of `members`, leave a unit of an XCD to somebody who completes a team
__host__ __device__ constexpr bool units_suffice(int queues, int members, int units) { return (long long)queues * (members - 1) < units; }

constexpr int SPIN_LIMIT = 1 << 23;   // polls of some 600 clocks: about two seconds
constexpr int SC1 = 16;               // cache policy of a load that goes past the L1

// a value from another lane of the row of 16 (data-parallel primitive); lanes past the row read 0
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int SHL = 0x100, SHR = 0x110, ROR = 0x120;   // shift to lower lanes, to higher ones, rotate

// the values of lanes l and l ^ 16 in row order
__device__ __forceinline__ v2u rows_of(float v) {
    const unsigned u = (unsigned)__float_as_int(v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return v2u{r[0], r[1]};
}

template <int DM, int MODE, bool FP8>
__global__ __launch_bounds__(512, 1) void team_kernel(const KArgs a) {
    constexpr bool ENC = MODE == MODE_ENC;
    typedef Cfg<DM> C;
    typedef typename Acc<FP8>::type acc_t;
    constexpr int D = C::D, NT = C::NT, TW = C::TW, CW = C::CW, KC = C::KC, KCF = C::KCF, NWG = C::NWG, TWW = C::TWW;
    constexpr int BPW = C::BPW, HB = C::HB, NP = C::NP;
    constexpr int BASE = 4 * KC * TW, SSTR = 4 * KC + 2 * TW;   // a quarter's stream: first feed-forward block of a layer, blocks of a step
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = lane & 31, g = lane >> 5;
    const int q = wave >> 1, iq0 = TWW * (wave & 1);   // the quarter of the width this wave's tiles lie in, the first one's number there

    // position `slot` of the launch belongs to workgroups slot % 8 + 8 (NWG (slot / 8) + m)
    const int m = (int)(blockIdx.x >> 3) % NWG;
    const int slot = ((int)(blockIdx.x >> 3) / NWG) * 8 + (int)(blockIdx.x & 7);
    int b = slot;
    if (a.leaf_index) {
        if (slot >= *a.leaf_count || slot >= a.n) return;
        b = __builtin_amdgcn_readfirstlane(a.leaf_index[slot]);
    }
    if ((unsigned)b >= (unsigned)a.n) return;
    if (a.active && !a.active[b]) return;

    uint8_t* const ws = a.team_ws + (size_t)slot * C::WS_BYTES;
    const __amdgpu_buffer_rsrc_t wsr = __builtin_amdgcn_make_buffer_rsrc(ws, 0, C::WS_BYTES, 0x00020000);
    unsigned* const flags = reinterpret_cast<unsigned*>(ws);
    const unsigned tag0 = (unsigned)__builtin_amdgcn_readfirstlane((int)flags[m]);   // layers of the launches before this one, modulo 2^32
    bool dead = false;                                           // this wave has given up waiting

    float* const xch = reinterpret_cast<float*>(lds + C::XCH_OFF);
    uint8_t* const act = lds + C::ACT_OFF;
    uint8_t* const hid = lds + C::HID_OFF;
    float* const tok = reinterpret_cast<float*>(lds + C::TOK_OFF);
    uint8_t* const ex = lds + C::EX_OFF;
    float* const qkv = reinterpret_cast<float*>(ex);
    const float* const gp = a.fparams + (size_t)4 * a.n_layers * C::PW_FLOATS;
    const int fq = 2 * (m & 1) + (wave >> 2), fh = wave & 3, fst = m >> 1;   // hidden tile 8 m + wave: its quarter, number there, step
    auto par = [&](int l, int quarter) { return reinterpret_cast<const float*>(lds + C::PAR_OFF + (l & 1) * C::PAR_BYTES) + quarter * C::P_FLOATS; };
    auto fetch_par = [&](int l, int quarter, bool first, bool rest) {   // of a quarter: part A, and what follows it
        const float* const src = a.fparams + ((size_t)quarter * a.n_layers + l) * C::PW_FLOATS;
        float* const dst = const_cast<float*>(par(l, quarter));
        if (first) dma(src, dst, C::A_FLOATS, lane);
        if (rest) {
            dma(src + C::A_FLOATS, dst + C::P_B, C::B_LDS_FLOATS, lane);
            dma(src + C::A_FLOATS + C::B_WSUM + m * CW, dst + C::P_WSUM, CW, lane);
            dma(src + C::A_FLOATS + C::B_BFF1 + 128 * fst, dst + C::P_BFF1, 128, lane);
        }
    };
    float* const fin = const_cast<float*>(par(a.l1, 0));   // the final norm's, after the last layer: [gamma][beta]
    static_assert(2 * D <= 4 * C::P_FLOATS, "they fit a copy");
    auto fetch_final = [&]() {
        dma(gp + C::G_NFG, fin, D, lane);
        dma(gp + C::G_NFB, fin + D, D, lane);
    };
    // block `idx` of layer l in a quarter's stream.  Buffer loads with the block's place in a scalar register: one
    // vector register of addresses for all of them (the stream is far below 4 GiB).
    const int stride_q = a.n_layers * BPW + HB + 1;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.wstream), 0, 4 * stride_q * BLOCK, 0x00020000);
    const int lane16 = lane * 16;
    auto load_block = [&](v4i (&w)[8], int quarter, int l, int idx) {
        const int at = (quarter * stride_q + l * BPW + idx) * BLOCK;
#pragma unroll
        for (int s = 0; s < 8; s++) w[s] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane16 + s % 4 * FRAG, at + s / 4 * 4 * FRAG, 0));
    };
    // Register sets of KC blocks.  Width 512, two: SA serves QKV, the second tile of the output projection, and the second
    // feed-forward matmul; SB the output projection and the first.  A set is filled as soon as it is free, an attention or an
    // exchange ahead of its use; SA for QKV between the vector instructions of LayerNorm 1 (spaced() below; 32 positions 322.6 ->
    // 319.5 us).  Width 256, three: SA QKV and the second feed-forward matmul, SB the output
    // projection, SC the first feed-forward matmul.  Each is filled where the wavefront has vector work to put between the loads
    // (spaced() below): SA and SB in LayerNorm 1, SC in the softmax, SA again in LayerNorm 2 -- or has nothing to do: SC by the
    // four that have no attention.  Filled at once, as soon as free: one position 82.3 us instead of 78.7.
    v4i SA[KC][8], SB[KC][8], SC[TWW == 1 ? KC : 1][8];
    auto& SF = [&]() -> auto& { if constexpr (TWW == 1) return SC; else return SB; }();
    const int hh = wave & 1, tq = wave >> 1;        // QKV: waves 0..5 take tile tq (Q, K, V) of head hh
    // the stream as waves 6 and 7 see it in fetch_qkv: empty, their loads move nothing (a branch around them could not be scheduled into)
    const __amdgpu_buffer_rsrc_t wq = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.wstream), 0, tq < 3 ? 4 * stride_q * BLOCK : 0, 0x00020000);
    const int head = 2 * m + hh, hq = head / TW, hi = head % TW;
    auto fetch_qkv = [&](int l) {
        const int at = tq < 3 ? (hq * stride_q + l * BPW + 3 * KC * hi + tq * KC) * BLOCK : 0, hop = tq < 3 ? 4 * FRAG : 0;
#pragma unroll
        for (int s = 0; s < 8 * KC; s++) SA[s / 8][s % 8] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wq, lane16 + s % 4 * FRAG, at + s / 4 * hop, 0));
    };
    auto fetch_out = [&](v4i (&w)[KC][8], int l, int i) {
#pragma unroll
        for (int c = 0; c < KC; c++) load_block(w[c], q, l, 3 * KC * TW + KC * (iq0 + i) + c);
    };
    auto fetch_ff1 = [&](int l) {
#pragma unroll
        for (int c = 0; c < KC; c++) load_block(SF[c], fq, l, BASE + fst * SSTR + KC * fh + c);
    };
    auto fetch_ff2 = [&](int l) {
#pragma unroll
        for (int i = 0; i < TWW; i++) load_block(SA[i], q, l, BASE + fst * SSTR + 4 * KC + (m & 1) * TW + iq0 + i);
    };
    static_assert(TWW <= KC, "the second feed-forward matmul's blocks fit the set");
    // `count` loads one at a time among the vector instructions of the code around (to the next barrier), `every` of those apart: the
    // unit takes a load in 16 clocks, so a set's eight at once, by all wavefronts, stop the wavefronts for a thousand.
    auto spaced = [&](auto every, auto count) {
#pragma unroll
        for (int i = 0; i < decltype(count)::value; i++) {
            __builtin_amdgcn_sched_group_barrier(0x002, decltype(every)::value, 0);   // vector instructions
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                        // a load
        }
    };
    auto product = [&](auto swap, const v4i (&w)[8], const uint8_t* from, acc_t acc) -> acc_t {
#pragma unroll
        for (int s = 0; s < 8; s++) acc = frag_mma<decltype(swap)::value>(w[s], *reinterpret_cast<const v4i*>(from + s * FRAG + lane * 16), acc);
        return acc;
    };
    const acc_t zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    // ---- rows: a wavefront owns the rows of tokens 4 wave .. + 3; a lane holds NP tiles of one of them, the half rg of the
    // accumulator layout.  Four neighbouring lanes are four tokens, which are neighbours in every buffer (64 bytes) ----
    const int row = 4 * wave + (lane & 3), rk = (lane >> 2) & 7, rg = lane >> 5;   // the token; tiles NP rk ..; the half
    const int rq = rk >> 1, ri = NP * (rk & 1);                                    // their quarter, the first one's number there
    // Sum of a row: tiles of a quarter as a tree, the quarters in order, the halves, as bf_args.h has it (v: the sum over the lane's
    // tiles).  A lane row of 16 holds two quarters: what lies in lanes 4 .. 15 comes to lanes 0 .. 3 and the result goes back.
    auto rowsum = [&](float v) -> float {
        v = v + dpp<SHL + 4>(v);
        const v2u r = rows_of(v);
        const float lo = __int_as_float(r[0]), hi = __int_as_float(r[1]);
        float s = ((lo + dpp<SHL + 8>(lo)) + hi) + dpp<SHL + 8>(hi);
        s = Rows<1>::sum({s});
        int u = __float_as_int(s);
        u = __builtin_amdgcn_update_dpp(u, u, SHR + 4, 0xf, 0x2, false);
        u = __builtin_amdgcn_update_dpp(u, u, SHR + 8, 0xf, 0xc, false);
        return __int_as_float(u);
    };
    // largest value of a row's 256-wide chunk
    auto chunkmax = [&](float v) -> float {
        v = vmax(v, dpp<ROR + 4>(v));
        v = vmax(v, dpp<ROR + 8>(v));
        v = Rows<1>::max({v});
        if constexpr (KC == 1) {
            const v2u r = rows_of(v);
            v = vmax(__int_as_float(r[0]), __int_as_float(r[1]));
        }
        return v;
    };
    // y = LayerNorm(x); gamma / beta: this lane's half of its first tile's parameters
    auto layernorm = [&](const float (&x)[NP][16], const float* gamma, const float* beta, float (&y)[NP][16]) {
        float ts[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            float acc = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) acc = acc + x[p][r];
            ts[p] = acc;
        }
        const float mean = rowsum(NP == 1 ? ts[0] : ts[0] + ts[NP - 1]) * (1.0f / D);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            float acc = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float d = x[p][r] - mean;
                acc = __builtin_fmaf(d, d, acc);
            }
            ts[p] = acc;
        }
        const float rstd = recip_sqrt(rowsum(NP == 1 ? ts[0] : ts[0] + ts[NP - 1]) * (1.0f / D) + a.eps);
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f ga = ldg4(gamma + 32 * p + 8 * j), be = ldg4(beta + 32 * p + 8 * j);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float d = x[p][4 * j + k] - mean;
                    y[p][4 * j + k] = __builtin_fmaf(d * rstd, ga[k], be[k]);
                }
            }
    };
    // quantise a row: its bytes go to the activation buffer as operand fragments, its scale(s) to the token table
    auto quantise = [&](const float (&y)[NP][16]) {
        float am = 0.0f;
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int r = 0; r < 16; r++) am = __builtin_fmaxf(am, __builtin_fabsf(y[p][r]));
        am = chunkmax(am);
        const float sa = row_scale<FP8>(am);
        if (rg == 0 && rk % (8 / KC) == 0) tok[rk / (8 / KC) * 32 + row] = sa;
        const Quot by = quot_by(sa);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            v4i w;
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = (int)quant4<FP8>(y[p][4 * j], y[p][4 * j + 1], y[p][4 * j + 2], y[p][4 * j + 3], by);
            *reinterpret_cast<v4i*>(act + (NP * rk + p) * FRAG + (rg * 32 + row) * 16) = w;
        }
    };
    auto scales = [&](float (&sa)[KC]) {   // of this lane's token, in the accumulator layout
#pragma unroll
        for (int c = 0; c < KC; c++) sa[c] = tok[c * 32 + t];
    };
    // wait until `met` holds of `count` flags and `tag`; `at`: this lane's flag
    constexpr Reached reached;
    constexpr Equal equal;
    auto wait_flags = [&](int at, int count, unsigned tag, auto met) {
        for (int spins = 0; !dead;) {
            unsigned f = tag;
            if (lane < count) f = __builtin_amdgcn_raw_buffer_load_b32(wsr, at * 4, 0, SC1);
            if (__all(met(f, tag))) break;
            if (++spins > SPIN_LIMIT) {
                dead = true;
                if (lane == 0) *a.team_gave_up = 1;
            }
            asm volatile("" ::: "memory");
        }
        asm volatile("" ::: "memory");
    };
    // this wave's piece is stored: let the L2 have it, then raise the flag
    auto raise_flag = [&](int at, unsigned tag) {
        wait_vm<0>();
        if (lane == 0 && !dead) __builtin_amdgcn_raw_buffer_store_b32(tag, wsr, 0, at * 4, 0);
    };
    // quad j of tile p of this wave's rows from the stream-shaped piece at `at`
    auto take = [&](int at, int p, int j) -> v4i {
        return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wsr, lane16, at + wave * C::ROWS_W + j * C::ROWS_Q + p * FRAG, SC1));
    };
    // where lane (t, g) of a tile in the accumulator layout has its place in a stream-shaped piece
    auto piece_at = [&](int tk, int half) { return (tk >> 2) * C::ROWS_W + (half * 32 + (tk & 3)) * 16; };
    auto tile_at = [&](int tile) { return tile % NP * FRAG + tile / NP * 64; };

    // ---- start: the board's words, then the first layer's parameters, which come while the rows that the words name are
    // asked for; its weights follow (all loads return in order) ----
    const unsigned own_word = ENC ? (a.taps.alive[(size_t)b * T + t] ? 0u : 0x800u) : a.boards[(size_t)b * T + t];
    const unsigned row_word = ENC ? 0u : a.boards[(size_t)b * T + row];
    const int ctrl = ENC ? 1 : a.control[b];
    int rp = ENC ? 0 : a.rep[b];
    rp = rp > 2 ? 2 : rp;
    __builtin_amdgcn_sched_barrier(0);
    if (a.l1 > a.l0) fetch_par(a.l0, q, !(wave & 1), wave & 1);
    else if (!ENC && wave == 4) fetch_final();
    __builtin_amdgcn_sched_barrier(0);

    // ---- embedding, or the caller's stream -------------------------------------------------------------
    // The rows that all tokens share (clock and repetition, added; the two of colour) come once, four bytes a thread, by way of
    // LDS: a load of sixteen bytes a lane takes the unit's path 16 clocks, and five rows for every token are 20 of them in each wave.
    float x[NP][16];
    const unsigned alive = (unsigned)__ballot(((own_word >> 11) & 1) == 0 && g == 0);
    if constexpr (ENC) {
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f v = stream_in(a.taps, ((size_t)b * T + row) * D + 32 * (NP * rk + p) + 4 * rg + 8 * j);
#pragma unroll
                for (int k = 0; k < 4; k++) x[p][4 * j + k] = v[k];
            }
    } else {
        float* const shared_rows = reinterpret_cast<float*>(ex);   // [clock + repetition][colour, bit 10 clear][set]
        static_assert(3 * D * 4 <= C::EX_BYTES && (D == 256 || D == 512), "shared rows");
        const int stm = ctrl < 0;
        int clock = (ctrl < 0 ? -ctrl : ctrl) - 1;
        clock = clock < 0 ? 0 : (clock > 100 ? 100 : clock);
        const int c = (int)threadIdx.x & (D - 1);
        const bool first = D == 512 || threadIdx.x < D, second = D == 512 || threadIdx.x >= D;   // whose share
        float once[4] = {};
        if (first) {
            once[0] = gp[C::G_CLOCK + clock * D + c];
            once[1] = gp[C::G_REP + rp * D + c];
        }
        if (second) {
            once[2] = gp[C::G_CT + stm * D + c];
            once[3] = gp[C::G_CT + (2 + stm) * D + c];
        }
        int ts = ((row_word >> 6) & 7) * 2 + ((row_word >> 9) & 1);
        ts = ts > 11 ? 11 : ts;
        v4f vs[NP][4], vt[NP][4];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int own = 32 * (NP * rk + p) + 4 * rg;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                vs[p][j] = ldg4(gp + C::G_SQ + (row_word & 63) * D + own + 8 * j);
                vt[p][j] = ldg4(gp + C::G_TS + ts * D + own + 8 * j);
            }
        }
        if (first) shared_rows[c] = once[0] + once[1];
        if (second) {
            shared_rows[D + c] = once[2];
            shared_rows[2 * D + c] = once[3];
        }
        lds_barrier();
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const float* const of = shared_rows + 32 * (NP * rk + p) + 4 * rg;
            const float* const colour = of + D + ((row_word >> 10) & 1) * D;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f vb = ldg4(of + 8 * j), vc = ldg4(colour + 8 * j);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    float v = vs[p][j][k] + vt[p][j][k];
                    v = v + vc[k];
                    x[p][4 * j + k] = v + vb[k];
                }
            }
        }
    }
#pragma unroll
    for (int p = 0; p < NP; p++) pin16(x[p]);   // has arrived, and with it the parameters, which were asked for before
    lds_barrier();

    for (int l = a.l0; l < a.l1; l++) {
        const unsigned tag = tag0 + (l - a.l0) + 1;
        const int lnext = l + 1 < a.l1 ? l + 1 : l;   // after the last layer its own weights come once more (and are not used)
        const float* const pq = par(l, q);                       // parameters of this wave's matmul tiles
        const float* const pr = par(l, rq) + 32 * ri + 4 * rg;   // of its rows: this lane's chain

        // ---- LayerNorm 1, quantise ---------------------------------------------------------------------
        {
            float y[NP][16];
            fetch_qkv(l);
            if constexpr (TWW == 1) fetch_out(SB, l, 0);
            layernorm(x, pr + C::A_LN1G, pr + C::A_LN1B, y);
            spaced(std::integral_constant<int, TWW == 1 ? 6 : 12>(), std::integral_constant<int, 16>());
            __builtin_amdgcn_sched_barrier(0);
            quantise(y);
        }
        lds_barrier();

        __builtin_amdgcn_sched_barrier(0);
        // ---- Q, K, V tiles of this member's heads ------------------------------------------------------
        // stored as [lane half g][register r odd][r / 8][token][r / 2 % 4], which is how the 16x16x4 operands are read
        if (tq < 3) {
            const float* const pA = par(l, hq);
            const float sw = pA[C::A_SW + tq * TW + hi];
            acc_t acc[KC];
            float v[16], sa[KC];
            scales(sa);
            if (tq < 2) {
#pragma unroll
                for (int c = 0; c < KC; c++) acc[c] = product(std::false_type(), SA[c], act + 8 * c * FRAG, zero);
                v4f bias[4];
                load_tile16(pA + (tq == 0 ? C::A_BQ : C::A_BK) + 32 * hi, g, bias);
#pragma unroll
                for (int r = 0; r < 16; r++) v[r] = chunk_sum<KC, false>(acc, r, sa) * sw + bias[r / 4][r % 4];
            } else {   // rows are tokens: the scale is that of token ch(r, g)
#pragma unroll
                for (int c = 0; c < KC; c++) acc[c] = product(std::true_type(), SA[c], act + 8 * c * FRAG, zero);
                const float bv = pA[C::A_BV + 32 * hi + t];
                v4f stok[KC][4];
#pragma unroll
                for (int c = 0; c < KC; c++) load_tile16(tok + 32 * c, g, stok[c]);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float st[KC];
#pragma unroll
                    for (int c = 0; c < KC; c++) st[c] = stok[c][r / 4][r % 4];
                    v[r] = chunk_sum<KC, false>(acc, r, st) * sw + bv;
                }
            }
            float* const to = qkv + (hh * 3 + tq) * 1024 + t * 4;
#pragma unroll
            for (int odd = 0; odd < 2; odd++)
#pragma unroll
                for (int iq = 0; iq < 2; iq++)
                    *reinterpret_cast<v4f*>(to + ((g * 2 + odd) * 2 + iq) * 128) = v4f{v[8 * iq + odd], v[8 * iq + 2 + odd], v[8 * iq + 4 + odd], v[8 * iq + 6 + odd]};
        }
        if constexpr (TWW > 1) {
            fetch_out(SB, l, 0);
            fetch_out(SA, l, 1);
        }
        lds_barrier();

        __builtin_amdgcn_sched_barrier(0);
        // ---- attention: head wave / 2, queries 16 (wave & 1) ... --------------------------------------------
        if (wave < 4) {
            const int ah = wave >> 1, qb = wave & 1, G = lane >> 4, c16 = lane & 15;
            const float* const from = qkv + ah * 3 * 1024 + ((G & 1) * 2 + (G >> 1)) * 256;   // operand k = G: lane half G & 1, register parity G >> 1
            auto operand = [&](int which, int row, float (&v)[8]) {
#pragma unroll
                for (int iq = 0; iq < 2; iq++) {
                    const v4f f = *reinterpret_cast<const v4f*>(from + which * 1024 + iq * 128 + row * 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[4 * iq + e] = f[e];
                }
            };
            // scores, transposed: lane = query; rows of the two key tiles are ordered so that lane row G's
            // register i holds key ch(2 i + G / 2, G % 2), the key it supplies to step i of P V
            float qv[8], kv[2][8];
            operand(0, 16 * qb + c16, qv);
#pragma unroll
            for (int u = 0; u < 2; u++) operand(1, ch(2 * (4 * u + (c16 & 3)) + (c16 >> 3), (c16 >> 2) & 1), kv[u]);
            v4f sc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int u = 0; u < 2; u++) sc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[u][i], qv[i], sc[u], 0, 0, 0);
            if constexpr (TWW == 1) fetch_ff1(l);
            float p[8];
            float mx = -__builtin_inff();
#pragma unroll
            for (int i = 0; i < 8; i++) {
                float s = sc[i / 4][i % 4] * 0.17677669529663687f;
                s = ((alive >> ch(2 * i + (G >> 1), G & 1)) & 1u) ? s : -__builtin_inff();
                p[i] = s;
                mx = vmax(mx, s);
            }
            mx = Rows<1>::max({mx});
            const v2u mr = rows_of(mx);
            mx = vmax(__int_as_float(mr[0]), __int_as_float(mr[1]));
            // a lane half's chain runs over r = 0 .. 15: even r in lane rows 0 and 1, odd r in rows 2 and 3
            float lsum = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                p[i] = exp_neg(p[i] - mx);
                const int iv = __float_as_int(p[i]);
                const auto both = __builtin_amdgcn_permlane32_swap(iv, iv, false, false);
                lsum = lsum + __int_as_float(both[0]);
                lsum = lsum + __int_as_float(both[1]);
            }
            const v2u lr = rows_of(lsum);
            const float rl = recip(__int_as_float(lr[0]) + __int_as_float(lr[1]));
            if constexpr (TWW == 1) spaced(std::integral_constant<int, 14>(), std::integral_constant<int, 8>());
            float vv[2][8];
#pragma unroll
            for (int u = 0; u < 2; u++) operand(2, 16 * u + c16, vv[u]);
            v4f oa[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float pi = p[i] * rl;
#pragma unroll
                for (int u = 0; u < 2; u++) oa[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[u][i], pi, oa[u], 0, 0, 0);
            }
            // channel 16 u + 4 G + e of query 16 qb + c16: register quad 2 u + G / 2 of lane (query, G % 2) of the tile
            const int tile = 2 * m + ah;
#pragma unroll
            for (int u = 0; u < 2; u++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, oa[u]), wsr,
                                                       piece_at(c16, G & 1) + (G >> 1) * C::ROWS_Q, C::WS_A + 4 * qb * C::ROWS_W + 2 * u * C::ROWS_Q + tile_at(tile), 0);
            raise_flag(C::FLAG_A + qb * NT + tile, tag);
        }
        if (wave >= 4) {
            // the other copy's last reads lie before the barriers above
            if (lnext != l) fetch_par(lnext, wave & 3, true, true);
            else if (!ENC && wave == 4) fetch_final();
            if constexpr (TWW == 1) fetch_ff1(l);
        }

        // ---- exchange A, output projection + residual --------------------------------------------------
        {
            float o[NP][16];
            wait_flags(C::FLAG_A + (wave >> 2) * NT + lane, NT, tag, reached);
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4f v = __builtin_bit_cast(v4f, take(C::WS_A, p, j));
#pragma unroll
                    for (int k = 0; k < 4; k++) o[p][4 * j + k] = v[k];
                }
            quantise(o);
            lds_barrier();
            float so[KC];
            scales(so);
#pragma unroll
            for (int i = 0; i < TWW; i++) {
                acc_t acc[KC];
#pragma unroll
                for (int c = 0; c < KC; c++) acc[c] = product(std::false_type(), i == 0 ? SB[c] : SA[c], act + 8 * c * FRAG, zero);
                if (TWW > 1 && i == 0) fetch_ff1(l);
                v4f bo[4];
                load_tile16(pq + C::A_BOUT + 32 * (iq0 + i), g, bo);
                const float sw = pq[C::A_SW + 3 * TW + iq0 + i];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v4f v;
#pragma unroll
                    for (int k = 0; k < 4; k++) v[k] = chunk_sum<KC, false>(acc, 4 * j + k, so) * sw + bo[j][k];
                    *reinterpret_cast<v4f*>(ex + (TWW * wave + i) * C::EX_TILE + j * FRAG + lane16) = v;
                }
            }
            lds_barrier();
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4f v = *reinterpret_cast<const v4f*>(ex + (NP * rk + p) * C::EX_TILE + j * FRAG + (rg * 32 + row) * 16);
#pragma unroll
                    for (int k = 0; k < 4; k++) x[p][4 * j + k] = x[p][4 * j + k] + v[k];
                }
        }

        __builtin_amdgcn_sched_barrier(0);
        // ---- LayerNorm 2, quantise, this member's chunk of the hidden row ---------------------------------
        {
            float y[NP][16];
            if constexpr (TWW == 1) fetch_ff2(l);
            layernorm(x, pr + C::P_B + C::B_LN2G, pr + C::P_B + C::B_LN2B, y);
            if constexpr (TWW == 1) spaced(std::integral_constant<int, 15>(), std::integral_constant<int, 8>());
            __builtin_amdgcn_sched_barrier(0);
            quantise(y);
        }
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
        float sh;
        if constexpr (TWW > 1) fetch_ff2(l);
        {
            const float* const pF = par(l, fq);
            acc_t acc[KC];
            float sa[KC];
            scales(sa);
#pragma unroll
            for (int c = 0; c < KC; c++) acc[c] = product(std::false_type(), SF[c], act + 8 * c * FRAG, zero);
            v4f b1[4];
            load_tile16(pF + C::P_BFF1 + 32 * fh, g, b1);
            const float sw1 = pF[C::P_B + C::B_SW + 4 * fst + fh];
            float hf[16], am = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                // int8: the ReLU is the saturation of the unsigned quantiser, the running maximum starts at 0
                float v = chunk_sum<KC, false>(acc, r, sa) * sw1 + b1[r / 4][r % 4];
                if constexpr (FP8) v = __builtin_fmaxf(v, 0.0f);
                hf[r] = v;
                am = __builtin_fmaxf(am, v);
            }
            xch[wave * 64 + lane] = am;
            lds_barrier();
            float mx = 0.0f;
#pragma unroll
            for (int w = 0; w < 8; w++) mx = __builtin_fmaxf(mx, xch[w * 64 + lane]);
            mx = Rows<1>::max({mx});
            sh = hidden_scale<FP8>(mx);
            const Quot by = quot_by(sh);
            v4i w;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (FP8) w[j] = (int)quant4<true>(hf[4 * j], hf[4 * j + 1], hf[4 * j + 2], hf[4 * j + 3], by);
                else w[j] = (int)(quant4_relu_u8(hf[4 * j], hf[4 * j + 1], hf[4 * j + 2], hf[4 * j + 3], by) ^ 0x80808080u);
            }
            *reinterpret_cast<v4i*>(hid + wave * FRAG + lane * 16) = w;
            lds_barrier();
        }

        __builtin_amdgcn_sched_barrier(0);
        // ---- second matmul over this member's chunk, exchange B ------------------------------------------
        {
#pragma unroll
            for (int i = 0; i < TWW; i++) {
                acc_t acc = zero;
                if constexpr (!FP8) {   // 128 * sum(w): the offset of the unsigned bytes stored as q - 128
                    v4i w0[4];
                    load_tile16i(pq + C::P_WSUM + 32 * (iq0 + i), g, w0);
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[r] = w0[r / 4][r % 4];
                }
                acc = product(std::false_type(), SA[i], hid, acc);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4i v = {accbits(acc, 4 * j), accbits(acc, 4 * j + 1), accbits(acc, 4 * j + 2), accbits(acc, 4 * j + 3)};
                    const int tile = TWW * wave + i;
                    if constexpr (C::TWO_STEPS) __builtin_amdgcn_raw_buffer_store_b128(v, wsr, lane16, C::piece_b(m, tile, j), 0);
                    else __builtin_amdgcn_raw_buffer_store_b128(v, wsr, piece_at(t, g), C::WS_B + m * C::ROWS + j * C::ROWS_Q + tile_at(tile), 0);
                }
                if constexpr (!C::TWO_STEPS)   // this member's own piece: through LDS
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        *reinterpret_cast<v4i*>(ex + wave * C::EX_TILE + j * FRAG + lane16) = v4i{accbits(acc, 4 * j), accbits(acc, 4 * j + 1), accbits(acc, 4 * j + 2), accbits(acc, 4 * j + 3)};
            }
            if constexpr (!C::TWO_STEPS) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the flag stands for it, too
            if (wave == 0 && g == 0) __builtin_amdgcn_raw_buffer_store_b32((unsigned)__float_as_int(sh), wsr, t * 4, C::scales_b(m), 0);
            raise_flag(C::flag_b(m, wave), tag);
            wait_flags(C::awaited_b(m, lane), C::FLAGS_B, tag, reached);
            if constexpr (C::TWO_STEPS) {
                // wave (i, j): quad j of tile i of this member's
                const int j = wave & 3, tile = C::tile_b(m, wave), tq2 = tile / TW, ti = tile % TW;
                v4i piece[NWG];
                float shc[NWG];
#pragma unroll
                for (int c = 0; c < NWG; c++) {
                    piece[c] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wsr, lane16, C::piece_b(c, tile, j), SC1));
                    shc[c] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(wsr, t * 4, C::scales_b(c), SC1));
                }
                const float* const pc = par(l, tq2) + C::P_B;
                const v4f b2 = ldg4(pc + C::B_BFF2 + 32 * ti + 8 * j + 4 * g);
                const float sw = pc[C::B_SW + 16 + ti];
                v4f upd;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    double o64 = (double)piece[0][k] * (double)shc[0];
#pragma unroll
                    for (int c = 1; c < NWG; c++) o64 = __builtin_fma((double)piece[c][k], (double)shc[c], o64);
                    upd[k] = (float)o64 * sw + b2[k];
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, upd), wsr, piece_at(t, g), C::WS_C + j * C::ROWS_Q + tile_at(tile), 0);
                raise_flag(C::FLAG_C + m * 8 + wave, tag);
                wait_flags(C::FLAG_C + lane, NWG * 8, tag, reached);
#pragma unroll
                for (int p = 0; p < NP; p++)
#pragma unroll
                    for (int jj = 0; jj < 4; jj++) {
                        const v4f v = __builtin_bit_cast(v4f, take(C::WS_C, p, jj));
#pragma unroll
                        for (int k = 0; k < 4; k++) x[p][4 * jj + k] = x[p][4 * jj + k] + v[k];
                    }
            } else {
                const float* const prB = par(l, rq) + C::P_B;
                float shc[NWG];
#pragma unroll
                for (int c = 0; c < NWG; c++) shc[c] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(wsr, row * 4, C::scales_b(c), SC1));
                // the others' pieces in order, and this member's own
                v4i piece[NWG - 1][4], own[4];
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int c = 0; c < NWG - 1; c++) piece[c][j] = take(C::WS_B + (c + (c >= m)) * C::ROWS, 0, j);
#pragma unroll
                for (int j = 0; j < 4; j++) own[j] = *reinterpret_cast<const v4i*>(ex + rk * C::EX_TILE + j * FRAG + (rg * 32 + row) * 16);
                const float sw = prB[C::B_SW + 16 + ri];
                auto sum_as = [&](auto member) {   // the sum runs over the members in order: one copy of it per place of the own piece
                    constexpr int M = decltype(member)::value;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        if constexpr (!FP8)   // its work stays in this copy, in the order of the loads (e4m3 is the faster without: 91.7 us against 92.9)
#pragma unroll
                            for (int c = 0; c < NWG - 1; c++) asm volatile("" : "+v"(piece[c][j]));
                        const v4f b2 = ldg4(pr + C::P_B + C::B_BFF2 + 8 * j);
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            double o64 = 0.0;
                            float upd = 0.0f;
#pragma unroll
                            for (int c = 0; c < NWG; c++) {
                                const int v = c == M ? own[j][k] : piece[c - (c > M)][j][k];
                                if constexpr (FP8) {
                                    const float part = (__int_as_float(v) * shc[c]) * prB[C::B_SW + 16 + ri * KCF + c];
                                    upd = c == 0 ? part : upd + part;
                                } else {
                                    const double full = (double)v, sc = (double)shc[c];
                                    o64 = c == 0 ? full * sc : __builtin_fma(full, sc, o64);
                                }
                            }
                            if constexpr (FP8) upd = upd + b2[k];
                            else upd = (float)o64 * sw + b2[k];
                            x[0][4 * j + k] = x[0][4 * j + k] + upd;
                        }
                    }
                    asm volatile("; %0" ::"n"(M));   // differs from copy to copy, or the compiler makes one of them and selects its operands, behind the last load
                };
                static_assert(C::TWO_STEPS || NWG == 4, "a copy per member");
                if (m == 0) sum_as(std::integral_constant<int, 0>());
                else if (m == 1) sum_as(std::integral_constant<int, 1>());
                else if (m == 2) sum_as(std::integral_constant<int, 2>());
                else sum_as(std::integral_constant<int, 3>());
            }
#pragma unroll
            for (int p = 0; p < NP; p++) {
                if (dead)
#pragma unroll
                    for (int r = 0; r < 16; r++) x[p][r] = __builtin_nanf("");
                pin16(x[p]);
            }
        }
    }
    if (wave == 0 && lane == 0) flags[m] = tag0 + (a.l1 - a.l0);

    if constexpr (ENC) {
        if (m == 0)
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    stream_out(a.taps, ((size_t)b * T + row) * D + 32 * (NP * rk + p) + 4 * rg + 8 * j,
                               v4f{x[p][4 * j], x[p][4 * j + 1], x[p][4 * j + 2], x[p][4 * j + 3]});
        return;
    }

    // ---- final norm and heads ------------------------------------------------------------------------------
    // Ten products of 16 rows of a head tile with 16 tokens, dealt out over the members' first wavefronts (each takes
    // a SIMD's matrix pipe and 32 KiB of head tile for itself): 0..7 the policy (tile, rows, tokens), 8 and 9 promotion
    // and value (the first rows of tile 2).
    const int job = wave * NWG + m;
    const int G = lane >> 4, c16 = lane & 15;
    // A head tile's fragments, HR of them in flight; the first ones now.  Lane (row, k) reads the fragment's lane of its row and of half
    // k % 2, from element k / 2 on, so that what it multiplies lies in places 0 and 2.  (The last lanes' reads end four bytes behind
    // the fragment, in the next one or the stream's block of padding.)
    constexpr int HR = 16;
    static_assert(8 * HB % HR == 0, "whole rounds");
    v4i hw[HR];
    auto load_head = [&](int ht, int rh, int f) {
        const int at = (ht * stride_q + a.n_layers * BPW) * BLOCK, lane_at = (16 * rh + c16 + 32 * (G & 1)) * 16 + 4 * (G >> 1);
        hw[f % HR] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane_at + f % 4 * FRAG, at + f / 4 * 4 * FRAG, 0));
    };
    auto load_first = [&](int ht, int rh) {
#pragma unroll
        for (int f = 0; f < HR; f++) load_head(ht, rh, f);
    };
    const int ht = job >> 2, rh = job < 8 ? (job >> 1) & 1 : 0, th = job & 1;   // job < 10: rows 16 rh .. of head tile ht, tokens 16 th ..
    if (job < 10) load_first(ht, rh);
    float hn[NP][16];
    const float* const gn = fin + 32 * NP * rk + 4 * rg;
    layernorm(x, gn, gn + D, hn);
    // as operand fragments (tile, quad)
    float* const hnb = reinterpret_cast<float*>(ex);
    auto publish = [&](const float (&v)[NP][16]) {
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                *reinterpret_cast<v4f*>(ex + (NP * rk + p) * C::EX_TILE + j * FRAG + (rg * 32 + row) * 16) = v4f{v[p][4 * j], v[p][4 * j + 2], v[p][4 * j + 1], v[p][4 * j + 3]};
    };
    publish(hn);
    if (lane == 0) xch[wave * 64] = dead ? 1.0f : 0.0f;   // a wave that has given up stands for its member
    lds_barrier();
#pragma unroll
    for (int w = 0; w < 8; w++) dead |= __builtin_amdgcn_readfirstlane(__float_as_int(xch[w * 64])) != 0;
    // (elements 0 and 2 of a register quad lie together, as do 1 and 3.)
    // Rows 16 rh .. of head tile `ht` times tokens 16 th ..: the chain of the 32x32x2 form, two of whose steps (four k) are
    // one step here.  Lane (row or token, k) takes element k / 2 and 2 + k / 2 of the fragment lane of half k % 2.
    auto head_product = [&](int ht, int rh, int th) -> v4f {
        int from = C::EX_OFF + (16 * th + c16 + 32 * (G & 1)) * 16 + 8 * (G >> 1);
        asm volatile("" : "+v"(from));   // one address register; the rest are the instructions' own offsets
        auto operand = [&](int f) { return *reinterpret_cast<const v2f*>(lds + from + f / 4 * C::EX_TILE + f % 4 * FRAG); };
        constexpr int EARLY = 8;   // operands come from LDS this many fragments early: the chain waits for its matrix steps only
        v2f h[EARLY];
#pragma unroll
        for (int f = 0; f < EARLY; f++) h[f] = operand(f);
        v4f acc = {0, 0, 0, 0};
#pragma unroll
        for (int f = 0; f < 8 * HB; f++) {
            const v4f w = __builtin_bit_cast(v4f, hw[f % HR]);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[0], h[f % EARLY][0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[2], h[f % EARLY][1], acc, 0, 0, 0);
            if (f + EARLY < 8 * HB) h[f % EARLY] = operand(f + EARLY);
            __builtin_amdgcn_sched_barrier(0);
            if (f + HR < 8 * HB) load_head(ht, rh, f + HR);
        }
        return acc;
    };
    auto marked = [&](const v4f& v) -> v4f {
        const float nan = __builtin_nanf("");
        return dead ? v4f{nan, nan, nan, nan} : v;
    };
    if (job < 8) {
        // policy: squares 32 ht + 16 rh + 4 G .. of token 16 th + c16, optional legal-move AND and argmax
        const int tk = 16 * th + c16, sq0 = 32 * ht + 16 * rh + 4 * G;
        unsigned long long mw = ~0ull;
        if (a.mask) mw = a.mask[(size_t)b * T + tk];
        const v4f hd = marked(head_product(ht, rh, th));
        float bv = -__builtin_inff(), v[4];
        int bi = 0x7fffffff;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const bool legal = (mw >> (sq0 + k)) & 1ull;
            v[k] = legal ? hd[k] : -__builtin_inff();
            if (legal && (bi == 0x7fffffff || v[k] > bv)) { bv = v[k]; bi = tk * 64 + sq0 + k; }
        }
        const size_t at = ((size_t)b * T + tk) * 64 + sq0;
        if (a.out_fp32) *reinterpret_cast<v4f*>((float*)a.policy + at) = v4f{v[0], v[1], v[2], v[3]};
        else *reinterpret_cast<v4h*>((_Float16*)a.policy + at) = v4h{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
        if (a.mask && a.best) {
            // larger, lowest index on ties; no move at all is worst
            auto merge = [&](float ov, int oi) {
                const bool take_ = oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi));
                bv = take_ ? ov : bv;
                bi = take_ ? oi : bi;
            };
            auto over_dpp = [&](auto ctrl) {
                constexpr int c = decltype(ctrl)::value;
                merge(dpp<c>(bv), __builtin_amdgcn_update_dpp(0, bi, c, 0xf, 0xf, true));
            };
            auto over_lanes_of_row = [&]() {   // xor 1, xor 2, the mirrored eight
                over_dpp(std::integral_constant<int, 0xb1>());
                over_dpp(std::integral_constant<int, 0x4e>());
                over_dpp(std::integral_constant<int, 0x141>());
            };
            over_lanes_of_row();
            over_dpp(std::integral_constant<int, 0x140>());
            auto over_swap = [&](auto swap) {   // both lanes get both values and keep the better one
                const auto v2 = swap(__float_as_int(bv)), i2 = swap(bi);
                bv = __int_as_float((int)v2[0]);
                bi = (int)i2[0];
                merge(__int_as_float((int)v2[1]), (int)i2[1]);
            };
            over_swap([](int v) { return __builtin_amdgcn_permlane16_swap(v, v, false, false); });
            over_swap([](int v) { return __builtin_amdgcn_permlane32_swap(v, v, false, false); });
            // the eight wavefronts' winners meet in member 0
            const unsigned tag = tag0 + (a.l1 - a.l0);
            if (lane == 0) __builtin_amdgcn_raw_buffer_store_b64(v2u{(unsigned)__float_as_int(bv), (unsigned)bi}, wsr, 0, C::WS_H + job * 16, 0);
            raise_flag(C::FLAG_H + job, tag);
            if (job == 0) {
                wait_flags(C::FLAG_H + lane, 8, tag, equal);
                const v2u w = __builtin_amdgcn_raw_buffer_load_b64(wsr, (lane & 7) * 16, C::WS_H, SC1);
                bv = __int_as_float((int)w[0]);
                bi = (int)w[1];
                over_lanes_of_row();
                if (lane == 0) a.best[b] = dead || bi == 0x7fffffff ? -1 : bi;
            }
        }
    }
    auto value_of = [&](const v4f& hd) -> float {
        if (dead) return __builtin_nanf("");   // (the functions below need not hand a NaN on)
        if (a.n_value == 1) return tanh_dev(hd[0]);
        const float r0 = hd[0], r1 = hd[1], r2 = hd[2];   // classes loss, draw, win
        const float mx = __builtin_fmaxf(__builtin_fmaxf(r0, r1), r2);
        const float e0 = exp_neg(r0 - mx), e1 = exp_neg(r1 - mx), e2 = exp_neg(r2 - mx);
        return (e2 - e0) / ((e0 + e1) + e2);
    };
    // rows 0..3 of head tile 2 are the promotion rows (lane row 0), rows 4.. the value rows (lane row 1)
    if (job == 8 || job == 9) {
        const v4f hd = marked(head_product(2, 0, th));
        const int tk = 16 * th + c16;
        if (G == 0) {
            const size_t at = ((size_t)b * T + tk) * 4;
            if (a.out_fp32) *reinterpret_cast<v4f*>((float*)a.promo + at) = hd;
            else *reinterpret_cast<v4h*>((_Float16*)a.promo + at) = v4h{(_Float16)hd[0], (_Float16)hd[1], (_Float16)hd[2], (_Float16)hd[3]};
        }
        if (a.vmode == 0 && G == 1 && tk == (ctrl < 0 ? 31 : 15)) a.value[b] = value_of(hd);
    }
    // pooled heads: the mean over the live tokens of the normalised stream (1), or the final norm of the mean of the
    // residual stream (2), through the value rows like a token; White's frame, so negated when Black is to move
    if (a.vmode != 0 && m == 0) {   // by all wavefronts of the member that has job 8
        // the mean runs over the tokens of a channel, a butterfly over the lanes of the accumulator layout: there and back
        if (a.vmode == 2) {
            lds_barrier();   // every wave has finished reading the normalised stream
            publish(x);
            lds_barrier();
        }
        const bool lv = (alive >> t) & 1u;
        const float cdiv = (float)(__builtin_popcount(alive) > 0 ? __builtin_popcount(alive) : 1);
        v4f pv[TWW][4];
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f s = *reinterpret_cast<const v4f*>(ex + (TWW * wave + i) * C::EX_TILE + j * FRAG + lane16);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    float v = lv ? s[k] : 0.0f;
#pragma unroll
                    for (int d = 16; d >= 1; d >>= 1) v = v + __shfl_xor(v, d);
                    pv[i][j][k] = v / cdiv;
                }
            }
        lds_barrier();
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) *reinterpret_cast<v4f*>(ex + (TWW * wave + i) * C::EX_TILE + j * FRAG + lane16) = pv[i][j];
        lds_barrier();
        if (a.vmode == 2) {
            float v[NP][16], hv[NP][16];
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4f s = *reinterpret_cast<const v4f*>(ex + (NP * rk + p) * C::EX_TILE + j * FRAG + (rg * 32 + row) * 16);
                    v[p][4 * j] = s[0]; v[p][4 * j + 2] = s[1]; v[p][4 * j + 1] = s[2]; v[p][4 * j + 3] = s[3];
                }
            layernorm(v, gn, gn + D, hv);
            lds_barrier();
            publish(hv);
            lds_barrier();
        }
        if (job == 8) {
            load_first(2, 0);
            const v4f hd = head_product(2, 0, 0);
            if (lane == 16) {
                const float v = value_of(hd);
                a.value[b] = ctrl > 0 ? v : -v;
            }
        }
    }
}

template <int DM, int MODE, bool FP8>
hipError_t launch_team(const KArgs& k, hipStream_t stream) {
    static std::atomic<unsigned long long> lds_set{0};
    typedef Cfg<DM> C;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipErrorInvalidDevice;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
    if (!(lds_set.load(std::memory_order_relaxed) & bit)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&team_kernel<DM, MODE, FP8>), hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
        if (e != hipSuccess) return e;
        lds_set.fetch_or(bit, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL((team_kernel<DM, MODE, FP8>), dim3((k.n + 7) / 8 * 8 * C::NWG), dim3(512), C::LDS_BYTES, stream, k);
    return hipGetLastError();
}

}  // namespace team
}  // namespace bf
