// The evaluator with TWO positions per workgroup of eight wavefronts (256-wide network).
//
// The decomposition is the eight-wavefront form of bf_board.hip.h -- wavefront (q, sub) owns
// tile 2q + sub of the model width, which is also its attention head, half of quarter q's tiles
// in every matmul, and reads its blocks out of the quarter's weight stream where they lie
// (board::block_at) -- but every wavefront does its share for two positions at once.  A weight
// fragment fetched from L2 into registers is then the A operand of two products, one per
// position, so a launch streams the weights once per pair of positions instead of once per
// position, and a wavefront has two independent instruction streams to fill its waits with.
// The quantised activations of both positions stay in LDS and are read as B operands at each
// product; the row statistics of both positions travel through the same exchange and the same
// workgroup barrier.  The arithmetic is that of the other kernels operation for operation, so
// the results are bit-identical to theirs.
//
// What bounds it (4096 positions, 8 layers, clocks of a SIMD per layer of some 54,000): the vector ALU's issue port, which
// retires additions, products and fused ones every 2.4 clocks from two wavefronts, everything else every 4.4, fp32 matrix
// steps (64 clocks, nothing beside them) and, of every int8 matrix step, 24 of its 33 clocks: together 45,000.  The rest
// are the thirteen exchanges of a layer, whose latencies both wavefronts of a SIMD wait out at the same time, and weights
// coming out of L2 in bursts.  So an exchange asks for everything at once, a row's statistics are computed once for both
// positions (Rows), addresses are made without vector instructions, and an accumulator is descaled without being converted: 1573 us -> 1463.
//
// NPOS = 1 is the same kernel with one position per workgroup: the latency form for launches of
// at most one workgroup per compute unit (each wavefront one tile of the width, every product
// issued under the previous product's epilogue, and the workgroups of an XCD warming the L2
// with the next layer's weights one layer ahead).
//
// LDS map (bytes): [xch: 3 slots x 2 positions x 8 waves x 64 floats] [act: the quantised row of the
// width, 8 KiB per position] [hid: the quantised hidden row, 32 KiB per position] [par: one
// copy of each quarter's side parameters, shared by its two wavefronts and both positions]
// [tok: the activation scale of every token of the row that feeds QKV, per position]
// [key: what masks every token's scores as a key, per position].
// During the heads the normalised stream of a position (32 KiB, fp32) overlays its hidden row.
//
// The e4m3 format widens each weight fragment to fp16 once for every position of the workgroup and keeps the row of the
// width widened in LDS; epilogues run under the next block's products here too (two pairs of accumulators, for which
// the weight ring gives up four places): 2143 us (TWIN) -> 1956.  The same vector ALU bounds it: a layer's 4,600 vector
// instructions per wavefront and 384 + 64 matrix steps are some 57,000 of 68,000 clocks.  Tried: chunks of the hidden row kept
// widened in LDS (-0.4 %: LDS then delivers as much as it can), two blocks side by side against each operand (-0.3 %).
#pragma once

#include "bf_heads.hip.h"

namespace bf {
namespace duo {

using board::block_at;
using board::BlockAt;
using board::frag_mma;
using board::lds;
using board::lds_barrier;
using board::tapbits;
using board::wait_vm;

template <bool FP8, int NP_>
struct Cfg : Layout<256> {
    static constexpr int NP = NP_, NW = 8;   // positions per workgroup (2; 1: the latency form), wavefronts
    static constexpr int XS = NP * NW * 64;               // floats of one exchange slot
    static constexpr int XCH_OFF = 0;
    static constexpr int ACT_OFF = XCH_OFF + 3 * XS * 4;
    // a position's quantised row of the width: operand bytes; in the e4m3 format widened to fp16 on
    // the way in (every e4m3 value is an fp16 value), so that the products read ready-made operands
    static constexpr int ACT_FRAG = FP8 ? 2 * FRAG : FRAG;
    static constexpr int ACT_P = NT * ACT_FRAG;
    static constexpr int HID_OFF = ACT_OFF + NP * ACT_P;
    static constexpr int HID_P = (F / 32) * FRAG;         // a position's hidden row
    static constexpr int PAR_OFF = HID_OFF + NP * HID_P;
    static constexpr int PWL_FLOATS = A_FLOATS + B_FLOATS;
    static constexpr int TOK_OFF = PAR_OFF + 4 * PWL_FLOATS * 4;   // activation scale of every token, per position
    static constexpr int KEY_OFF = TOK_OFF + NP * 32 * 4;          // what is added to the scores of every key: 0, or -inf for a dead token
    static constexpr int USED_BYTES = KEY_OFF + NP * 32 * 4;
    // The one-position form serves launches of at most one workgroup per compute unit: asking for
    // more than half of a unit's LDS keeps the dispatcher from placing two of them on one unit
    // while another unit stays empty.
    static constexpr int LDS_BYTES = NP == 1 && USED_BYTES < 81 * 1024 ? 81 * 1024 : USED_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget: one workgroup per compute unit");
    static_assert(NT * 4 * FRAG <= HID_P, "normalised stream overlay");

    static constexpr int RING = NP == 2 ? 8 : 12;   // weight fragments (four registers each) in flight or in use
    // L2 warm-up (see warm_l2 in the kernel): touches of a wavefront per layer; the line of the quarters' streams that touch j of a lane
    // falls on, and whether there is one
    static constexpr int WARM = NP == 1 ? 2 : 0, LAYER_LINES = Layout<256>::BPW * BLOCK / 128;   // lines of a layer, per quarter
    static __host__ __device__ constexpr int warm_line(int j, int block, int blocks, int wave, int lane) {
        return ((j * ((blocks + 7) >> 3) + (block >> 3)) * 8 + wave) * 64 + lane;
    }
    static __host__ __device__ constexpr bool warms(int line, int blocks) { return blocks > 24 && blocks <= 256 && line < 4 * LAYER_LINES; }
    // Loads that every wavefront has under way behind the first layer's parameters, whatever the launch: the ring's first fill.  A touch is
    // none of them, since a launch, or a wavefront of it, may have none.  (tests/test_duo_start.py goes through all of them.)
    static constexpr int BEHIND_PARAMETERS = RING;
};

// one 16-deep step on operands already widened to fp16; int8 builds never call it
template <bool SWAP>
__device__ __forceinline__ v16f f16_step(const v8h& w, const v8h& act, const v16f& acc) {
    return SWAP ? __builtin_amdgcn_mfma_f32_32x32x16_f16(act, w, acc, 0, 0, 0)
                : __builtin_amdgcn_mfma_f32_32x32x16_f16(w, act, acc, 0, 0, 0);
}
template <bool SWAP>
__device__ __forceinline__ v16i f16_step(const v8h&, const v8h&, const v16i& acc) { return acc; }

template <int MODE, bool FP8, bool PROF = false, int NPOS = 2>
__device__ __forceinline__ void evaluate(const KArgs& a, const int block, const int blocks) {   // workgroup `block` of `blocks`
    constexpr bool TAPS = MODE == MODE_TAPS, ENC = MODE == MODE_ENC;
    typedef Cfg<FP8, NPOS> C;
    static_assert(NPOS == 1 || NPOS == 2, "positions per workgroup");
    typedef typename Acc<FP8>::type acc_t;
    constexpr int NP = C::NP, D = C::D, F = C::F, NT = C::NT, TW = C::TW, CW = C::CW, KCF = C::KCF;
    constexpr int STEPS = C::STEPS, BPW = C::BPW, HB = C::HB;
    constexpr int NB = BPW / 2;      // weight blocks a wave consumes per layer
    constexpr int HT = 2;            // hidden tiles a wave computes per feed-forward step
    // Weight fragments in flight or in use, and steps between the LDS fetch of an operand fragment and its use
    // (4096 positions: 1496 us with one, 1498 with three, as a SIMD's other wavefront covers the latency; the one-position form at 100
    // positions: 118.3 and 116.7; encoder-only, two positions, 512 of them: 179.0, and 179.8 with a register spilled)
    constexpr int RING = C::RING, AHEAD = NP == 2 && ENC ? 1 : 3;
    constexpr bool SUBN = !FP8 && !TAPS;   // how accumulators are descaled, see descale() (tapped accumulators are stored as they are)
    constexpr int XS = C::XS, PS = C::NW * 64;   // floats of an exchange slot; of one position's part of it
    static_assert(C::KC == 1 && STEPS == TW && KCF == 2 * STEPS, "the 256-wide network");
    static_assert(8 % (AHEAD + 1) == 0, "an operand's place must not depend on the product");
    static_assert((8 * NB) % RING == 0, "a fragment's place in the ring must not depend on the layer");
    static_assert(RING <= 8 * HB, "the first prefetches of the heads stay inside the head blocks");
    static_assert(board::block_at_covers_layer<1, TW, 2, BPW, true>(), "block_at must enumerate a layer's blocks exactly once");

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = wave & 3, sub = wave >> 2;
    const int tile = TW * q + sub;   // the tile of the width (and the head) this wave owns
    const int t = lane & 31, g = lane >> 5;

    // the positions of this workgroup: its own NP slots of the launch, or those entries of the
    // compacted leaf list.  A slot without a position (past the end, skipped, not in this launch)
    // computes its neighbour's position again and stores nothing; a workgroup without any position
    // leaves before the first barrier.
    int bp[NP];
    bool live[NP];
    {
        int cnt = a.n, first = (NP == 1 ? a.single_from : 0) + NP * block;
        if (a.leaf_index) {
            cnt = *a.leaf_count < a.n ? *a.leaf_count : a.n;   // the list has n entries whatever the count says
            if (a.list_split) {
                if (NP == 1) first += cnt - round_rest(cnt);
                else cnt -= round_rest(cnt);
            }
        }
        bool any = false;
        int some = 0;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int j = first + p;
            int b = j;
            bool ok = j < cnt;
            if (a.leaf_index) {
                b = ok ? __builtin_amdgcn_readfirstlane(a.leaf_index[j]) : 0;
                ok = ok && (unsigned)b < (unsigned)a.n;
            }
            if (ok && a.active) ok = a.active[b] != 0;
            bp[p] = ok ? b : 0;
            live[p] = ok;
            if (ok) { any = true; some = b; }
        }
        if (!any) return;
#pragma unroll
        for (int p = 0; p < NP; p++)
            if (!live[p]) bp[p] = some;
    }
    const int nl_run = a.l1 - a.l0;
    // Phase accounting (PROF builds only): the shader clock is read at phase boundaries and the
    // cycles since the previous mark are charged to a slot; the time spent inside workgroup
    // barriers is summed separately (and is also contained in the enclosing phases).
    unsigned long long ph[N_PHASES];
    unsigned long long t_mark = 0, t_begin = 0, t_sync = 0;
    if constexpr (PROF) {
#pragma unroll
        for (int i = 0; i < N_PHASES; i++) ph[i] = 0;
        t_mark = t_begin = __builtin_readcyclecounter();
    }
#define BF_PHASE(slot)                                                    \
    do {                                                                  \
        if constexpr (PROF) {                                             \
            __builtin_amdgcn_sched_barrier(0); /* nothing is scheduled across the mark */ \
            const unsigned long long now_ = __builtin_readcyclecounter(); \
            __builtin_amdgcn_sched_barrier(0);                            \
            ph[slot] += now_ - t_mark;                                    \
            t_mark = now_;                                                \
        }                                                                 \
    } while (0)
    auto barrier = [&]() {
        if constexpr (PROF) {
            const unsigned long long t0_ = __builtin_readcyclecounter();
            lds_barrier();
            t_sync += __builtin_readcyclecounter() - t0_;
        } else {
            lds_barrier();
        }
    };

    // the lane's offsets, as opaque values: known bits would let the compiler make a base register out of every sum
    // of them with a constant instead of using the instructions' own offsets
    int lane16 = lane * 16, lane4 = lane * 4;
    asm volatile("" : "+v"(lane16));
    asm volatile("" : "+v"(lane4));
    float* const xch = reinterpret_cast<float*>(lds + C::XCH_OFF);
    const float* const xlane = reinterpret_cast<const float*>(lds + C::XCH_OFF + lane4);
    uint8_t* const hid = lds + C::HID_OFF;
    uint8_t* const act = lds + C::ACT_OFF;
    float* const tok = reinterpret_cast<float*>(lds + C::TOK_OFF);
    float* const key = reinterpret_cast<float*>(lds + C::KEY_OFF);
    const bool par_owner = sub == 0;
    float* const pA = reinterpret_cast<float*>(lds + C::PAR_OFF) + q * C::PWL_FLOATS;
    float* const pB = pA + C::A_FLOATS;
    // LDS addresses that a layer uses once or twice are made where they are used (one vector addition): the empty asm
    // keeps the compiler from hoisting them all out of the layer loop, where two dozen of them hold a register each
    // that the operand and weight rings need.
    auto here = [&](const void* at) -> uint8_t* {
        int off = (int)(static_cast<const uint8_t*>(at) - lds);
        asm volatile("" : "+s"(off));
        return lds + off;
    };
    auto here_f = [&](const float* at) -> float* { return reinterpret_cast<float*>(here(at)); };
    const uint8_t* const wsrc =
        a.wstream + ((size_t)q * ((size_t)a.n_layers * BPW + HB + 1) + (size_t)a.l0 * BPW) * BLOCK;   // uniform
    // the quarter's stream as a buffer: a load's address is a uniform offset and the lane's own, with no vector
    // arithmetic and no address registers
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wsrc), 0, ((a.n_layers - a.l0) * BPW + HB + 1) * BLOCK, 0x00027000);
    const __amdgpu_buffer_rsrc_t pbuf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.fparams + (size_t)q * a.n_layers * C::PW_FLOATS), 0, a.n_layers * C::PW_FLOATS * 4, 0x00027000);
    // `nfloats` of the quarter's side parameters, from float `at` on, straight into LDS
    auto fetch_par = [&](int at, float* dst, int nfloats) {
        uint8_t* const d = reinterpret_cast<uint8_t*>(dst);
        const int bytes = nfloats * 4, full = bytes / FRAG, rem = (bytes % FRAG) / 16;
#pragma unroll
        for (int i = 0; i <= full; i++)
            if (i < full || lane < rem)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(pbuf, (__attribute__((address_space(3))) void*)(d + i * FRAG), 16, lane16, at * 4 + i * FRAG, 0, 0);
    };
    const float* const gp = a.fparams + (size_t)4 * a.n_layers * C::PW_FLOATS;

    // What descaled accumulators start from: the integer whose bits are the smallest normal float (see descale())
    acc_t start = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (SUBN)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            int v = 0x00800000;
            asm volatile("" : "+v"(v));   // kept, not made anew for every product
            start[i] = v;
        }
    // The weight fragments in flight: a ring of RING registers-of-four, refilled one by one.  What the loads cost is their rate
    // out of L2 and not their latency (a build without them runs 8 % shorter, one whose loads all hit L1 as well): two
    // positions, 4096 of them: 8 places 1463 us, 12 with the sixteen registers of `start` beside them 1489 (14 spilled), without
    // 1481.  One position: 12 places 120.3 us, 16 120.7, 24 128.6 (spilled).  Fragment `fseq` of the
    // quarter's stream into place `at`.
    v4i frt[RING];
    auto load_frag = [&](int fseq, int at) {
        const int src = fseq * FRAG;
        frt[at] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, lane16, src, 0));
    };
    // the wave's ff-th fragment of the layer whose stream starts at block `base` (ff may run into the following layer,
    // whose stream starts at block `next`)
    auto fetch_frag = [&](int ff, int base, int next) {
        const int n = ff / 8;
        const BlockAt at = block_at<1, TW, 2, true>(n % NB);
        load_frag(8 * ((n < NB ? base : next) + at.a + sub * at.b) + ff % 8, ff % RING);
    };

    // L2 warm-up for launches of one wave of workgroups (NP == 1): such a launch moves through the
    // layers in step, so every first touch of a weight line would be an L2 miss that all the
    // workgroups behind that L2 wait for.  The workgroups of an XCD (dispatched round-robin, so
    // block / 8 numbers them) each touch a share of the lines of a layer's blocks one layer ahead,
    // one dword per 128-byte line; the values are never used.  A hint only: a share that nobody
    // touches (workgroups that left early, another dispatch order) costs time, not correctness.
    // Below four workgroups per XCD the touches cover too little to pay for the loads they delay
    // (loads return in order), above one workgroup per compute unit the launch is not in step.
    constexpr int WARM = C::WARM, LAYER_LINES = C::LAYER_LINES;
    int warm[WARM > 0 ? WARM : 1] = {};
    auto warm_l2 = [&](int blk0) {
        if constexpr (WARM > 0) {
#pragma unroll
            for (int j = 0; j < WARM; j++) {
                const int line = C::warm_line(j, block, blocks, wave, lane);
                if (C::warms(line, blocks)) {
                    const int qq = line / LAYER_LINES, off = line % LAYER_LINES;
                    warm[j] = *reinterpret_cast<const int*>(
                        a.wstream + ((size_t)qq * ((size_t)a.n_layers * BPW + HB + 1) + (size_t)blk0) * BLOCK + (size_t)off * 128);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto warm_done = [&]() {   // the touches have long returned: retire their registers
        if constexpr (WARM > 0) {
#pragma unroll
            for (int j = 0; j < WARM; j++) asm volatile("" ::"v"(warm[j]));
        }
    };

    // Row sum over the width for both positions: a wave's 16 values form one chain from zero, the
    // two tile sums of a quarter are added, then the four quarter sums in order.  One exchange slot
    // per call site, so that a fast wave's next partial cannot overwrite what a slow wave still
    // reads: between two uses of a slot lies at least one other workgroup barrier.
    // An exchange is a chain of latencies that both wavefronts of a SIMD wait out together, so everything a
    // wave reads behind the barrier is asked for at once, before the first value is used.
    auto xsum2 = [&](const float (&part)[NP], int slot) -> float {
#pragma unroll
        for (int p = 0; p < NP; p++) here_f(xch + slot * XS + p * PS + wave * 64)[lane] = part[p];
        barrier();
        float s[NP][8], out[NP];
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int w = 0; w < C::NW; w++) s[p][w] = xlane[slot * XS + p * PS + w * 64];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < NP; p++) out[p] = (((s[p][0] + s[p][4]) + (s[p][1] + s[p][5])) + (s[p][2] + s[p][6])) + (s[p][3] + s[p][7]);
        return Rows<NP>::sum(out);
    };
    // Largest value of the rows over waves [W0, W0 + 1, ...]: a wave publishes, for two positions, one value a row
    // (Rows<2>::max, half the traffic of the lanes' own), for one position its lanes' own.
    auto xmax_put = [&](const float (&am)[NP], int at) { here_f(xch + at + wave * 64)[lane] = NP == 2 ? Rows<NP>::max(am) : am[0]; };
    auto xmax_row = [&](float m) -> float {
        if constexpr (NP == 2) return m;
        const float v[1] = {m};
        return Rows<1>::max(v);
    };
    auto layernorm2_by = [&](const float (&x)[NP][16], auto gamma, auto beta, float (&y)[NP][16]) {   // gamma(j), beta(j): of register quad j
        float part[NP], mean[NP], rstd[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            float acc = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) acc = acc + x[p][r];
            part[p] = acc;
        }
        Rows<NP>::each(xsum2(part, 0) * (1.0f / D), mean);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            float acc = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float d = x[p][r] - mean[p];
                acc = __builtin_fmaf(d, d, acc);
            }
            part[p] = acc;
        }
        Rows<NP>::each(recip_sqrt(xsum2(part, 1) * (1.0f / D) + a.eps), rstd);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const v4f ga = gamma(j), be = beta(j);
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float d = x[p][4 * j + k] - mean[p];
                    y[p][4 * j + k] = __builtin_fmaf(d * rstd[p], ga[k], be[k]);
                }
        }
    };
    auto layernorm2 = [&](const float (&x)[NP][16], const float* gamma, const float* beta, float (&y)[NP][16]) {
        layernorm2_by(x, [&](int j) { return ldg4(gamma + 8 * j + 4 * g); }, [&](int j) { return ldg4(beta + 8 * j + 4 * g); }, y);
    };
    // signed quantiser of both positions' rows: one scale per row; this wave's bytes go to the
    // position's activation buffer, from which every wave reads its B operands
    auto quant_exchange2 = [&](const float (&y)[NP][16], float (&sa)[NP], float (&ex)[NP], int8_t* tap, const size_t (&tap_row)[NP], bool publish_scales) {
        float am[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            am[p] = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) am[p] = __builtin_fmaxf(am[p], __builtin_fabsf(y[p][r]));
        }
        xmax_put(am, 2 * XS);
        barrier();
        float mw[8];
#pragma unroll
        for (int w = 0; w < C::NW; w++) mw[w] = xlane[2 * XS + w * 64];
        const float sr = row_scale<FP8>(xmax_row(vmax3(vmax3(mw[0], mw[1], mw[2]), vmax3(mw[3], mw[4], mw[5]), vmax(mw[6], mw[7]))));
        if constexpr (SUBN) {   // the scale in two parts: its significand times 2^126 (NaN: NaN), its exponent and 23
            const int bits = __float_as_int(sr);
            Rows<NP>::each(__builtin_fmaf(sr, 0.0f, __int_as_float((bits & 0x007fffff) | 0x7e800000)), sa);
            Rows<NP>::each(__int_as_float((bits >> 23) - 127 + 23), ex);
        } else Rows<NP>::each(sr, sa);
        if (publish_scales && wave == 0 && lane < 32 * NP) here_f(tok)[lane] = sr;
        const Quot br = quot_by(sr);
        float hi[NP], lo[NP];
        Rows<NP>::each(br.hi, hi);
        Rows<NP>::each(br.lo, lo);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const Quot by = {hi[p], lo[p]};
            v4i w;
#pragma unroll
            for (int j = 0; j < 4; j++)
                w[j] = (int)quant4<FP8>(y[p][4 * j], y[p][4 * j + 1], y[p][4 * j + 2], y[p][4 * j + 3], by);
            if constexpr (FP8) {
                const v2l wl = __builtin_bit_cast(v2l, w);
#pragma unroll
                for (int h = 0; h < 2; h++)
                    *reinterpret_cast<v8h*>(here(act + p * C::ACT_P + (2 * tile + h) * FRAG) + lane16) = e4m3x8_as_f16(wl[h]);
            } else {
                *reinterpret_cast<v4i*>(here(act + p * C::ACT_P + tile * FRAG) + lane16) = w;
            }
            if (TAPS && tap && live[p])
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *reinterpret_cast<int*>(tap + (tap_row[p] * T + t) * D + 32 * tile + 8 * j + 4 * g) = w[j];
        }
        barrier();
    };
    const uint8_t* const act0 = act + lane16;
    const uint8_t* const hid0 = hid + lane16;
    auto ldsfrag = [&](const uint8_t* p) -> v4i { return *reinterpret_cast<const v4i*>(p); };

    // An encoder-only launch (tap table with `alive`): the residual stream comes in through x_in, the
    // token mask through `alive`, the stream after the last layer goes out through resid_last, and
    // there are no board words and no heads.
    const bool enc_only = ENC || (TAPS && a.taps.alive != nullptr);
    // ---- embedding (this wave's tile, both positions) ----------------------------------------------
    // Loads return in order, so what the first layer's weights would hold up is asked for in front of them: the words, then the rows they
    // name.  A unit takes a 16-byte load of 64 lanes in 16 clocks, and five rows for every token are 40 of them in each wave; so
    // the rows that a position's tokens share (clock and repetition, added; the two of colour) come once, four bytes a thread, by way of LDS.
    // Phase 12.9 k -> 10.1 k ticks; 300 positions 168.2 -> 167.0 us, 100 113.8 -> 113.0, 4096 1411 -> 1404, e4m3 1891 -> 1881.
    // (Parameters, touches and the weights stand behind branches, where the compiler cannot count them, and it waits for all of them:
    // the last position's rows are still used only once the first weights are there.)
    float x[NP][16];
    unsigned alive[NP], word[NP];
    int ctrl[NP], rp[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int b = bp[p];
        word[p] = enc_only ? (a.taps.alive[(size_t)b * T + t] ? 0u : 0x800u) : a.boards[(size_t)b * T + t];
        ctrl[p] = enc_only ? 1 : a.control[b];
        rp[p] = enc_only ? 0 : a.rep[b];
    }
    const bool given = ENC || (TAPS && a.taps.x_in);   // the caller's stream
    float* const shared_rows = reinterpret_cast<float*>(hid);   // per position: [clock + repetition][colour, bit 10 clear][set], D floats each
    float once[4];
    v4f vs[NP][4], vt[NP][4];
    if (!given) {
        const int c = (int)threadIdx.x & (D - 1), p = NP == 2 ? sub : 0;
        const int stm = (p ? ctrl[NP - 1] : ctrl[0]) < 0, cw = p ? ctrl[NP - 1] : ctrl[0];
        int clock = (cw < 0 ? -cw : cw) - 1;
        clock = clock < 0 ? 0 : (clock > 100 ? 100 : clock);
        const int rep = p ? rp[NP - 1] : rp[0], r2 = rep > 2 ? 2 : rep;
        once[0] = gp[C::G_CLOCK + clock * D + c];
        once[1] = gp[C::G_REP + r2 * D + c];
        once[2] = gp[C::G_CT + stm * D + c];
        once[3] = gp[C::G_CT + (2 + stm) * D + c];
#pragma unroll
        for (int q_ = 0; q_ < NP; q_++) {
            int ts = ((word[q_] >> 6) & 7) * 2 + ((word[q_] >> 9) & 1);
            ts = ts > 11 ? 11 : ts;
            load_tile16(gp + C::G_SQ + (word[q_] & 63) * D + 32 * tile, g, vs[q_]);
            load_tile16(gp + C::G_TS + ts * D + 32 * tile, g, vt[q_]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- start the first layer's parameters and the weight stream ----------------------------------
    if (nl_run > 0) {
        if (par_owner) {
            fetch_par(a.l0 * C::PW_FLOATS, pA, C::A_FLOATS);
            fetch_par(a.l0 * C::PW_FLOATS + C::A_FLOATS, pB, C::B_FLOATS);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < RING; j++) fetch_frag(j, 0, BPW);
        warm_l2(a.l0 * BPW);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!given) {
        float* const to = shared_rows + (NP == 2 ? sub : 0) * 3 * D + ((int)threadIdx.x & (D - 1));
        if (NP == 2 || sub == 0) {
            to[0] = once[0] + once[1];
            to[D] = once[2];
            to[2 * D] = once[3];
        }
        barrier();
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int b = bp[p];
        alive[p] = (unsigned)__ballot(((word[p] >> 11) & 1) == 0 && g == 0);
        if (wave == 0 && g == 0) key[p * 32 + t] = ((word[p] >> 11) & 1) == 0 ? 0.0f : -__builtin_inff();
        if (given) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f v = stream_in(a.taps, ((size_t)b * T + t) * D + 32 * tile + 8 * j + 4 * g);
#pragma unroll
                for (int k = 0; k < 4; k++) x[p][4 * j + k] = v[k];
            }
        } else {
            const float* const of = shared_rows + p * 3 * D + 32 * tile;
            v4f vb[4], vc[4];
            load_tile16(of, g, vb);
            load_tile16(of + D + ((word[p] >> 10) & 1) * D, g, vc);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    float v = vs[p][j][k] + vt[p][j][k];
                    v = v + vc[j][k];
                    x[p][4 * j + k] = v + vb[j][k];
                }
        }
        if (TAPS && a.taps.embed && live[p])
#pragma unroll
            for (int r = 0; r < 16; r++) a.taps.embed[((size_t)b * T + t) * D + 32 * tile + ch(r, g)] = x[p][r];
    }

    wait_vm<C::BEHIND_PARAMETERS>();   // the parameters have landed: what was asked for after them may not (published to the quarter's other wave by the next barrier)
    warm_done();
    BF_PHASE(PH_EMBED);

    for (int l = a.l0; l < a.l1; l++) {
        const int li = l - a.l0;
        size_t bl[NP];   // tap rows
#pragma unroll
        for (int p = 0; p < NP; p++) bl[p] = (size_t)bp[p] * nl_run + li;
        const int lnext = l + 1 < a.l1 ? l + 1 : l;   // after the last layer the same layer is fetched again (and never used)
        const int lbase = li * BPW, lfollow = (lnext - a.l0) * BPW;
        // One position's product with the wave's k-th block of this layer: eight 32-deep steps against
        // the operand row whose fragment 0 is at BSRC (lane offset included), each fragment fetched
        // from LDS one step ahead.  The last position refills a fragment's place in the ring as soon as it has
        // consumed it, with the fragment RING further on, so every place is in flight or full across the phases
        // between products (attention, the LayerNorms).
        // BETWEEN(s) runs after step s has been issued: an eighth of the previous product's epilogue,
        // which the vector ALU works through while the matrix pipe runs; nothing is scheduled across
        // the end of a step.  One position per workgroup: the epilogue starts a step later, so that its first value is there
        // when it is asked for (200 positions 112.5 -> 111.8 us; two positions, whose other wavefront has work meanwhile: no change).
        // The operand fragments come from LDS AHEAD steps early, also across the products of a phase: in its last
        // steps a product fetches the first operands of the next one (at NEXT, if there is one whose operands are
        // written already: MORE).  BF_DUO_OPERANDS opens a phase with the first product's.
#define BF_DUO_OPERANDS(BSRC)                                                                        \
    v4i ops_[AHEAD + 1];                                                                             \
    _Pragma("unroll") for (int u_ = 0; u_ < AHEAD; u_++) ops_[u_] = ldsfrag((BSRC) + u_ * FRAG)
#define BF_DUO_CHAIN(SWAP, k, p, BSRC, MORE, NEXT, INIT, R, BETWEEN)                                 \
    do {                                                                                             \
        const uint8_t *const b_ = (BSRC), *const n_ = (NEXT);                                        \
        (R) = (INIT);                                                                                \
        _Pragma("unroll") for (int s_ = 0; s_ < 8; s_++) {                                           \
            if (s_ + AHEAD < 8) ops_[(s_ + AHEAD) % (AHEAD + 1)] = ldsfrag(b_ + (s_ + AHEAD) * FRAG); \
            else if (MORE) ops_[(s_ + AHEAD) % (AHEAD + 1)] = ldsfrag(n_ + (s_ + AHEAD - 8) * FRAG);   \
            (R) = frag_mma<SWAP>(frt[(8 * (k) + s_) % RING], ops_[s_ % (AHEAD + 1)], (R));           \
            if (NP == 2) BETWEEN(s_);                                                                \
            else if (s_ > 0) BETWEEN(s_ - 1);                                                        \
            if (NP == 1 && s_ == 7) BETWEEN(7);                                                      \
            __builtin_amdgcn_sched_barrier(0);                                                       \
            if ((p) == NP - 1) fetch_frag(8 * (k) + s_ + RING, lbase, lfollow);                      \
        }                                                                                            \
    } while (0)
        // e4m3: the positions' products with the wave's k-th block, step by step.  A weight fragment is widened to
        // fp16 once and multiplied with every position's operands; these come from LDS already widened
        // (A16: the row of the width) or as bytes (the hidden row), position p's STRIDE bytes on.  Each accumulator
        // sees its sixteen 16-deep steps in order, as in the other kernels.  BETWEEN(s): an eighth of the
        // previous product's epilogues, as above.
#define BF_DUO_PRODUCT_F8(SWAP, k, A16, B, STRIDE, R, BETWEEN)                                       \
    do {                                                                                             \
        const uint8_t* const b_ = (B);                                                               \
        constexpr int PER_ = (A16) ? 2 : 1;   /* operand fragments of a step */                      \
        v4i cur_[NP], nxt_[NP];                                                                      \
        _Pragma("unroll") for (int p_ = 0; p_ < NP; p_++) {                                          \
            (R)[p_] = zero;                                                                          \
            cur_[p_] = ldsfrag(b_ + p_ * (STRIDE));                                                  \
        }                                                                                            \
        _Pragma("unroll") for (int s_ = 0; s_ < 8; s_++) {                                           \
            const v2l wl_ = __builtin_bit_cast(v2l, frt[(8 * (k) + s_) % RING]);                      \
            _Pragma("unroll") for (int h_ = 0; h_ < 2; h_++) {                                       \
                const bool new_ = h_ == 1 || (A16);                                                  \
                const int u_ = PER_ * s_ + (h_ + 1) * PER_ / 2;   /* the fragment after this one */  \
                if (new_ && u_ < 8 * PER_)                                                           \
                    _Pragma("unroll") for (int p_ = 0; p_ < NP; p_++) nxt_[p_] = ldsfrag(b_ + p_ * (STRIDE) + u_ * FRAG); \
                const v8h wh_ = e4m3x8_as_f16(wl_[h_]);                                              \
                _Pragma("unroll") for (int p_ = 0; p_ < NP; p_++) {                                  \
                    v8h ah_;                                                                         \
                    if (A16) ah_ = __builtin_bit_cast(v8h, cur_[p_]);                                \
                    else ah_ = e4m3x8_as_f16(__builtin_bit_cast(v2l, cur_[p_])[h_]);                 \
                    (R)[p_] = f16_step<SWAP>(wh_, ah_, (R)[p_]);                                     \
                    if (new_) cur_[p_] = nxt_[p_];                                                   \
                }                                                                                    \
            }                                                                                        \
            BETWEEN(s_);                                                                             \
            __builtin_amdgcn_sched_barrier(0);                                                       \
            fetch_frag(8 * (k) + s_ + RING, lbase, lfollow);                                         \
        }                                                                                            \
    } while (0)
        const acc_t zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        // An accumulator a times its row's scale s and its channel's w: fl(fl(a s) w).  int8: the sum of a matmul of the width is
        // below 2^22, and the products start at 2^23, so that what comes out, 2^23 + a, is the bit pattern of the float
        // (2^23 + a) 2^-149: up to 2^24 the bits of subnormal and smallest normal floats count linearly.  One fused operation takes
        // the offset off and multiplies: with s = m 2^e, fma(x, m 2^126, -m) = fl(a m) 2^-23, exactly rounded as fl(a s) is, and
        // 2^(e + 23) goes into w (ldexp, once a tile).  That takes the place of a conversion, 4.4 clocks, and a product: 4096
        // positions 1481 -> 1463 us, 200 positions 115.2 -> 113.6, same bits for 2^-149 <= s w < 2^104:
        // above, w 2^(e + 23) overflows (infinite results, and NaN for a = 0) though fl(fl(a s) w) may be finite yet; below, it
        // loses bits to the subnormal range.  Rows without a largest value, NaN, stay NaN.
        auto descale = [&](const acc_t& ac, int e, float s, float off, float w) -> float {
            if constexpr (SUBN) return __builtin_fmaf(__int_as_float(accbits(ac, e)), s, off) * w;
            else return accf(ac, e) * s * w;
        };
        auto offsets = [&](const float (&sa)[NP], float (&off)[NP]) {
#pragma unroll
            for (int p = 0; p < NP; p++) off[p] = SUBN ? sa[p] * -0x1p-126f : 0.0f;
        };
        auto scaled = [&](float w, const float (&ex)[NP], float (&to)[NP]) {
#pragma unroll
            for (int p = 0; p < NP; p++) to[p] = SUBN ? __builtin_ldexpf(w, __float_as_int(ex[p])) : w;
        };
        auto none = [&](int) {};

        // ---- LayerNorm 1, quantise, exchange -----------------------------------------------------------
        float sa[NP], ex[NP];
        {
            float y[NP][16];
            layernorm2(x, here_f(pA + C::A_LN1G + 32 * sub), here_f(pA + C::A_LN1B + 32 * sub), y);
            quant_exchange2(y, sa, ex, TAPS ? a.taps.qa_qkv : nullptr, bl, true);
        }
        // the quarter's feed-forward parameters of this layer (the first layer's came with the start)
        if (par_owner && li > 0) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            fetch_par(l * C::PW_FLOATS + C::A_FLOATS, pB, C::B_FLOATS);
        }
        BF_PHASE(PH_LN1);

        // ---- attention: this wave's head, both positions ------------------------------------------------
        float o[NP][16];
        {
            float qf[NP][16], kf[NP][16], vf[NP][16];
            const float* const sw3 = here_f(pA + C::A_SW + sub);
            const float swq = sw3[0], swk = sw3[TW], swv = sw3[2 * TW];
            const float bv = here_f(pA + C::A_BV + 32 * sub)[t];
            float off[NP], wq[NP], wk[NP];
            offsets(sa, off);
            scaled(swq, ex, wq);
            scaled(swk, ex, wk);
            acc_t acc[2];   // product n of a sequence uses accumulator n & 1; the previous one's epilogue runs under it
            v4f bq[4], bk[4], stok[NP][4];
            // the epilogues, two accumulator registers at a time (slice s of eight)
            auto epi_q = [&](int p, int s, const acc_t& ac) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) {
                    qf[p][e] = descale(ac, e, sa[p], off[p], wq[p]) + bq[e / 4][e % 4];
                    if (TAPS && a.taps.acc_qkv && live[p])
                        a.taps.acc_qkv[(bl[p] * T + t) * 3 * D + 32 * tile + ch(e, g)] = tapbits<false>(ac, e);
                }
            };
            auto epi_k = [&](int p, int s, const acc_t& ac) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) {
                    kf[p][e] = descale(ac, e, sa[p], off[p], wk[p]) + bk[e / 4][e % 4];
                    if (TAPS && a.taps.acc_qkv && live[p])
                        a.taps.acc_qkv[(bl[p] * T + t) * 3 * D + D + 32 * tile + ch(e, g)] = tapbits<false>(ac, e);
                }
            };
            // V tile: rows are tokens, so the activation scale is that of token ch(e, g)
            auto epi_v = [&](int p, int s, const acc_t& ac) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) {
                    vf[p][e] = accf(ac, e) * stok[p][e / 4][e % 4] * swv + bv;
                    if (TAPS && a.taps.acc_qkv && live[p])
                        a.taps.acc_qkv[(bl[p] * T + ch(e, g)) * 3 * D + 2 * D + 32 * tile + t] = tapbits<false>(ac, e);
                }
            };
            auto epi_qkv = [&](int tq, int p, int s, const acc_t& ac) {
                if (tq == 0) epi_q(p, s, ac);
                else if (tq == 1) epi_k(p, s, ac);
                else epi_v(p, s, ac);
            };
            // A SIMD favours its older wavefront, which then waits at the next exchange for a partner that has the SIMD to
            // itself: the younger one goes first here, the older one in the attention behind (4096 positions -1.3 to
            // -2.9 %, e4m3 -1.8 %; first in the attention too: +5 to +10 %; in other phases: nothing)
            if (sub) __builtin_amdgcn_s_setprio(2);
            load_tile16(here_f(pA + C::A_BQ + 32 * sub), g, bq);
            if constexpr (FP8) {
                // e4m3: a block's two products share the widening of its weight fragments; the epilogues of both
                // positions run under the next block's
                acc_t pair[2][NP];
                BF_DUO_PRODUCT_F8(false, 0, true, act0, C::ACT_P, pair[0], none);
                load_tile16(here_f(pA + C::A_BK + 32 * sub), g, bk);
                auto with_q = [&](int s) {
#pragma unroll
                    for (int p = 0; p < NP; p++) epi_q(p, s, pair[0][p]);
                };
                BF_DUO_PRODUCT_F8(false, 1, true, act0, C::ACT_P, pair[1], with_q);
#pragma unroll
                for (int p = 0; p < NP; p++) load_tile16(here_f(tok + 32 * p), g, stok[p]);
                auto with_k = [&](int s) {
#pragma unroll
                    for (int p = 0; p < NP; p++) epi_k(p, s, pair[1][p]);
                };
                BF_DUO_PRODUCT_F8(true, 2, true, act0, C::ACT_P, pair[0], with_k);
#pragma unroll
                for (int s = 0; s < 8; s++)
#pragma unroll
                    for (int p = 0; p < NP; p++) epi_v(p, s, pair[0][p]);
            } else {
                // Q, K, V blocks in turn, each for every position: 3 NP products
                BF_DUO_OPERANDS(act0);
#pragma unroll
                for (int n = 0; n < 3 * NP; n++) {
                    const int tq = n / NP, p = n % NP;
                    if (n == NP) load_tile16(here_f(pA + C::A_BK + 32 * sub), g, bk);
                    if (tq == 2) load_tile16(here_f(tok + 32 * p), g, stok[p]);
                    auto between = [&](int s) {
                        if (n > 0) epi_qkv((n - 1) / NP, (n - 1) % NP, s, acc[(n - 1) & 1]);
                    };
                    const uint8_t* const next = act0 + (n + 1) % NP * C::ACT_P;
                    if (tq == 2) BF_DUO_CHAIN(true, 2, p, act0 + p * C::ACT_P, n + 1 < 3 * NP, next, zero, acc[n & 1], between);
                    else BF_DUO_CHAIN(false, tq, p, act0 + p * C::ACT_P, n + 1 < 3 * NP, next, start, acc[n & 1], between);
                }
#pragma unroll
                for (int s = 0; s < 8; s++) epi_v(NP - 1, s, acc[(3 * NP - 1) & 1]);
            }
            __builtin_amdgcn_s_setprio(0);
            BF_PHASE(PH_QKV);
            if (l + 1 < a.l1) warm_l2((l + 1) * BPW);   // the sets are full and the next weight wait is an attention away
            v16f sc[NP];   // scores, transposed: lane = query token, register r = key ch(r, g)
            auto scores = [&](int p) {
                sc[p] = v16f{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < 16; r++) sc[p] = BF_F32MMA(kf[p][r], qf[p][r], sc[p]);
            };
            float pr[NP][16], rl[NP];
            auto softmax = [&](int p) {
                float mx = -__builtin_inff();
                v4f kb[4];
                load_tile16(here_f(key + 32 * p), g, kb);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    // scaled and masked in one operation: adding 0 changes nothing, a dead key's -inf (or what an infinite
                    // score makes of it, NaN) loses in the maximum and has probability 0
                    pr[p][r] = __builtin_fmaf(sc[p][r], 0.17677669529663687f, kb[r / 4][r % 4]);
                    mx = __builtin_fmaxf(mx, pr[p][r]);
                }
                const float mx1[1] = {mx};
                mx = Rows<1>::max(mx1);
                float lsum = 0.0f;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    pr[p][r] = exp_neg(pr[p][r] - mx);
                    lsum = lsum + pr[p][r];
                }
                const float ls1[1] = {lsum};
                rl[p] = recip(Rows<1>::sum(ls1));
            };
            auto weigh = [&](int p) {
                v16f oa = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < 16; r++) oa = BF_F32MMA(vf[p][r], pr[p][r] * rl[p], oa);
#pragma unroll
                for (int r = 0; r < 16; r++) o[p][r] = oa[r];
                pin16(o[p]);
            };
#pragma unroll
            for (int p = 0; p < NP; p++) { scores(p); softmax(p); weigh(p); }
            BF_PHASE(PH_ATTN);
        }

        // ---- output projection + residual (this wave's tile) --------------------------------------------
        {
            float so[NP], eo[NP], off[NP], wo[NP];
            quant_exchange2(o, so, eo, TAPS ? a.taps.qa_out : nullptr, bl, false);
            acc_t acc[2];
            v4f bo[4];
            load_tile16(here_f(pA + C::A_BOUT + 32 * sub), g, bo);
            const float sw = *here_f(pA + C::A_SW + 3 * TW + sub);
            offsets(so, off);
            scaled(sw, eo, wo);
            auto epi_o = [&](int p, int s, const acc_t& ac) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) {
                    x[p][e] = x[p][e] + (descale(ac, e, so[p], off[p], wo[p]) + bo[e / 4][e % 4]);
                    if (TAPS && a.taps.acc_out && live[p])
                        a.taps.acc_out[(bl[p] * T + t) * D + 32 * tile + ch(e, g)] = tapbits<false>(ac, e);
                }
            };
            if constexpr (FP8) {
                BF_DUO_PRODUCT_F8(false, 3, true, act0, C::ACT_P, acc, none);
                if (NP > 1)
#pragma unroll
                    for (int s = 0; s < 8; s++) epi_o(0, s, acc[0]);
            } else {
                BF_DUO_OPERANDS(act0);
#pragma unroll
                for (int p = 0; p < NP; p++) {
                    auto between = [&](int s) {
                        if (p > 0) epi_o(p - 1, s, acc[(p - 1) & 1]);
                    };
                    BF_DUO_CHAIN(false, 3, p, act0 + p * C::ACT_P, p + 1 < NP, act0 + C::ACT_P, start, acc[p & 1], between);
                }
            }
#pragma unroll
            for (int s = 0; s < 8; s++) epi_o(NP - 1, s, acc[(NP - 1) & 1]);
        }
        BF_PHASE(PH_OUT);

        // ---- feed-forward ---------------------------------------------------------------------------------
        {
            float y[NP][16];
            layernorm2(x, here_f(pB + C::B_LN2G + 32 * sub), here_f(pB + C::B_LN2B + 32 * sub), y);
            quant_exchange2(y, sa, ex, TAPS ? a.taps.qa_ff1 : nullptr, bl, false);
        }
        // the attention-phase parameters are dead for both waves of the quarter: fetch the next layer's
        if (par_owner) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            fetch_par(lnext * C::PW_FLOATS, pA, C::A_FLOATS);
        }
        BF_PHASE(PH_LN2);
        // First matmul, step by step: each step's two 256-wide chunks are quantised as soon as the step
        // is complete (a chunk spans a pair of quarters); the whole quantised hidden row of both
        // positions stays in LDS.  int8: unsigned, bytes stored as q - 128 for the signed MFMA.
        float sh[NP][KCF];
#pragma unroll
        for (int st = 0; st < STEPS; st++) {
            BF_DUO_OPERANDS(act0);
            float hf[NP][HT][16];
            float am[NP];
#pragma unroll
            for (int p = 0; p < NP; p++) am[p] = 0.0f;
            acc_t acc[2], pair[2][NP];   // e4m3: a block's products at a time
            v4f b1[HT][4];
            float off[NP], sw1[HT][NP];
            offsets(sa, off);
            auto epi_f = [&](int i, int p, int s, const acc_t& ac) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) {
                    // the ReLU is in the hidden quantiser's saturation, and the running maximum starts at 0,
                    // so negative values need no clamp here
                    const float v = descale(ac, e, sa[p], off[p], sw1[i][p]) + b1[i][e / 4][e % 4];
                    hf[p][i][e] = v;
                    am[p] = __builtin_fmaxf(am[p], v);
                    if (TAPS && a.taps.acc_ff1 && live[p])
                        a.taps.acc_ff1[(bl[p] * T + t) * F + 512 * st + 128 * q + 32 * (HT * sub + i) + ch(e, g)] = tapbits<false>(ac, e);
                }
            };
#pragma unroll
            for (int i = 0; i < HT; i++) {
                load_tile16(here_f(pB + C::B_BFF1 + 128 * st + 32 * (HT * sub + i)), g, b1[i]);
                scaled(*here_f(pB + C::B_SW + 4 * st + HT * sub + i), ex, sw1[i]);
                if constexpr (FP8) {
                    auto with_f = [&](int s) {
                        if (i > 0)
#pragma unroll
                            for (int p = 0; p < NP; p++) epi_f(i - 1, p, s, pair[(i - 1) & 1][p]);
                    };
                    BF_DUO_PRODUCT_F8(false, 4 + HT * st + i, true, act0, C::ACT_P, pair[i & 1], with_f);
                } else {
#pragma unroll
                    for (int p = 0; p < NP; p++) {
                        const int n = NP * i + p;   // product number within the step; the previous one's epilogue runs under it
                        auto between = [&](int s) {
                            if (n > 0) epi_f((n - 1) / NP, (n - 1) % NP, s, acc[(n - 1) & 1]);
                        };
                        BF_DUO_CHAIN(false, 4 + HT * st + i, p, act0 + p * C::ACT_P, n + 1 < NP * HT, act0 + (p + 1) % NP * C::ACT_P, start, acc[n & 1],
                                     between);
                    }
                }
            }
            if constexpr (FP8)
#pragma unroll
                for (int s = 0; s < 8; s++)
#pragma unroll
                    for (int p = 0; p < NP; p++) epi_f(HT - 1, p, s, pair[(HT - 1) & 1][p]);
            else
#pragma unroll
                for (int s = 0; s < 8; s++) epi_f(HT - 1, NP - 1, s, acc[(NP * HT - 1) & 1]);
            // the maxima of consecutive steps go through different exchange slots
            const int xs = (st & 1) ? 0 : 2 * XS;
            xmax_put(am, xs);
            barrier();
            float hi[NP], lo[NP];
            {
                float mw[8], sc[2];
#pragma unroll
                for (int w = 0; w < C::NW; w++) mw[w] = xlane[xs + w * 64];
#pragma unroll
                for (int c = 0; c < 2; c++) {   // chunk c: quarters 2c and 2c + 1 (hidden values are >= 0)
                    float each[NP];
                    sc[c] = hidden_scale<FP8>(xmax_row(vmax(vmax3(mw[2 * c], mw[2 * c + 1], mw[2 * c + 4]), mw[2 * c + 5])));
                    Rows<NP>::each(sc[c], each);
#pragma unroll
                    for (int p = 0; p < NP; p++) sh[p][2 * st + c] = each[p];
                }
                const Quot br = quot_by(q < 2 ? sc[0] : sc[1]);
                Rows<NP>::each(br.hi, hi);
                Rows<NP>::each(br.lo, lo);
            }
#pragma unroll
            for (int p = 0; p < NP; p++) {
                const Quot by = {hi[p], lo[p]};
#pragma unroll
                for (int i = 0; i < HT; i++) {
                    v4i w;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        unsigned u;
                        if constexpr (FP8) u = quant4_relu_e4m3(hf[p][i][4 * j], hf[p][i][4 * j + 1], hf[p][i][4 * j + 2], hf[p][i][4 * j + 3], by);
                        else u = quant4_relu_u8(hf[p][i][4 * j], hf[p][i][4 * j + 1], hf[p][i][4 * j + 2], hf[p][i][4 * j + 3], by);
                        if (TAPS && a.taps.qa_ff2 && live[p])
                            *reinterpret_cast<unsigned*>(a.taps.qa_ff2 + (bl[p] * T + t) * F + 512 * st + 128 * q + 32 * (HT * sub + i) + 8 * j + 4 * g) = u;
                        w[j] = (int)(FP8 ? u : (u ^ 0x80808080u));
                    }
                    *reinterpret_cast<v4i*>(here(hid + p * C::HID_P + (16 * st + 4 * q + HT * sub + i) * FRAG) + lane16) = w;
                }
            }
        }
        barrier();   // the whole hidden row of both positions is in LDS
        BF_PHASE(PH_FF1);
        // Second matmul: this wave's output tile over the KCF k-chunks in turn; each chunk's block
        // serves both positions.  int8: the accumulator starts at 128 * sum(w), the offset of the
        // unsigned bytes stored as q - 128; the sums over the chunks are float64 (e4m3: fp32).
        {
            double o64[NP][16];
            float o32[NP][16];
            acc_t acc[2], pair[2][NP];
            acc_t init = zero;
            BF_DUO_OPERANDS(hid0);
            float sw2[KCF];   // e4m3: one weight scale per k-chunk
            if constexpr (FP8)
#pragma unroll
                for (int cc = 0; cc < KCF; cc++) sw2[cc] = here_f(pB + C::B_SW + 16 + sub * KCF)[cc];
            auto epi_2 = [&](int cc, int p, int s, const acc_t& ac) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) {
                    if constexpr (FP8) {
                        const float part = (accf(ac, e) * sh[p][cc]) * sw2[cc];
                        o32[p][e] = cc == 0 ? part : o32[p][e] + part;
                    } else {
                        const double sc = (double)sh[p][cc];
                        const int full = accbits(ac, e);
                        o64[p][e] = cc == 0 ? (double)full * sc : __builtin_fma((double)full, sc, o64[p][e]);
                    }
                    if (TAPS && a.taps.acc_ff2 && live[p])
                        a.taps.acc_ff2[((bl[p] * KCF + cc) * T + t) * D + 32 * tile + ch(e, g)] = accbits(ac, e);
                }
            };
#pragma unroll
            for (int cc = 0; cc < KCF; cc++) {
                if constexpr (FP8) {
                    auto with_2 = [&](int s) {
                        if (cc > 0)
#pragma unroll
                            for (int p = 0; p < NP; p++) epi_2(cc - 1, p, s, pair[(cc - 1) & 1][p]);
                    };
                    BF_DUO_PRODUCT_F8(false, 4 + HT * STEPS + cc, false, hid0 + 8 * cc * FRAG, C::HID_P, pair[cc & 1], with_2);
                } else {
#pragma unroll
                    for (int p = 0; p < NP; p++) {
                        const int n = NP * cc + p, cn = (n + 1) / NP, pn = (n + 1) % NP;
                        if (p == 0) {
                            v4i w0[4];
                            load_tile16i(here_f(pB + C::B_WSUM + cc * CW + 32 * sub), g, w0);
#pragma unroll
                            for (int j = 0; j < 4; j++)
#pragma unroll
                                for (int k = 0; k < 4; k++) init[4 * j + k] = w0[j][k];
                        }
                        auto between = [&](int s) {
                            if (n > 0) epi_2((n - 1) / NP, (n - 1) % NP, s, acc[(n - 1) & 1]);
                        };
                        BF_DUO_CHAIN(false, 4 + HT * STEPS + cc, p, hid0 + p * C::HID_P + 8 * cc * FRAG,
                                     cn < KCF, hid0 + pn * C::HID_P + 8 * cn * FRAG, init, acc[n & 1], between);
                    }
                }
            }
            if constexpr (FP8)
#pragma unroll
                for (int s = 0; s < 8; s++)
#pragma unroll
                    for (int p = 0; p < NP; p++) epi_2(KCF - 1, p, s, pair[(KCF - 1) & 1][p]);
            else
#pragma unroll
                for (int s = 0; s < 8; s++) epi_2(KCF - 1, NP - 1, s, acc[(NP * KCF - 1) & 1]);
            v4f b2[4];
            load_tile16(here_f(pB + C::B_BFF2 + 32 * sub), g, b2);
            const float sw = *here_f(pB + C::B_SW + 16 + sub);
#pragma unroll
            for (int p = 0; p < NP; p++) {
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        float upd;
                        if constexpr (FP8) upd = o32[p][4 * j + k] + b2[j][k];
                        else upd = (float)o64[p][4 * j + k] * sw + b2[j][k];
                        x[p][4 * j + k] = x[p][4 * j + k] + upd;
                    }
                pin16(x[p]);
            }
        }
        BF_PHASE(PH_FF2);
        warm_done();
#undef BF_DUO_OPERANDS
#undef BF_DUO_CHAIN
#undef BF_DUO_PRODUCT_F8
        if (TAPS && a.taps.resid)
#pragma unroll
            for (int p = 0; p < NP; p++)
                if (live[p])
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        a.taps.resid[(bl[p] * T + t) * D + 32 * tile + ch(r, g)] = x[p][r];
    }
    if constexpr (ENC) {
#pragma unroll
        for (int p = 0; p < NP; p++)
            if (live[p])
#pragma unroll
                for (int j = 0; j < 4; j++)
                    stream_out(a.taps, ((size_t)bp[p] * T + t) * D + 32 * tile + 8 * j + 4 * g,
                               v4f{x[p][4 * j], x[p][4 * j + 1], x[p][4 * j + 2], x[p][4 * j + 3]});
        return;
    }
    if (TAPS && a.taps.resid_last)
#pragma unroll
        for (int p = 0; p < NP; p++)
            if (live[p])
#pragma unroll
                for (int r = 0; r < 16; r++)
                    a.taps.resid_last[((size_t)bp[p] * T + t) * D + 32 * tile + ch(r, g)] = x[p][r];
    if (enc_only) return;   // the same for every wave of the launch

    // ---- final norm and heads --------------------------------------------------------------------------
    Heads<NP, HB, RING> heads(a, BPW, lane, wave, bp, live, ctrl, C::HID_OFF, C::HID_P);
    // the final norm's parameters, a quarter's worth of exchanges ahead of their use
    v4f nfg[4], nfb[4];
    load_tile16(gp + C::G_NFG + 32 * tile, g, nfg);
    load_tile16(gp + C::G_NFB + 32 * tile, g, nfb);
    heads.ask();
    __builtin_amdgcn_sched_barrier(0);
    auto final_norm = [&](const float (&of)[NP][16], float (&y)[NP][16]) {
        layernorm2_by(of, [&](int j) { return nfg[j]; }, [&](int j) { return nfb[j]; }, y);
    };
    float hn[NP][16];
    final_norm(x, hn);
    auto publish = [&](int p, const float (&v)[16]) { heads.publish(p, tile, v); };
#pragma unroll
    for (int p = 0; p < NP; p++) {
        if (TAPS && a.taps.normed && live[p])
#pragma unroll
            for (int r = 0; r < 16; r++)
                a.taps.normed[((size_t)bp[p] * T + t) * D + 32 * tile + ch(r, g)] = hn[p][r];
        publish(p, hn[p]);
    }
    barrier();
    heads.products();
    BF_PHASE(PH_HEADS);
    heads.store(xch + 2 * XS, barrier);   // the exchange slot no row sum uses
    // ---- pooled value heads (reference brokefish/nn/model.py:576-617) --------------------------------
    // The value row is the mean over the live tokens of the normalised stream ("pooled", mode 1) or
    // the final LayerNorm of the mean of the residual stream ("prenorm", mode 2); it goes through
    // the value rows of head tile 2 like a token, and the result is in White's frame, so it is
    // negated when Black is to move.
    if (a.vmode != 0) {
        float pv[NP][16], hv[NP][16];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const bool lv = (alive[p] >> t) & 1u;
            const float cdiv = (float)(__builtin_popcount(alive[p]) > 0 ? __builtin_popcount(alive[p]) : 1);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                float v = lv ? (a.vmode == 1 ? hn[p][r] : x[p][r]) : 0.0f;
#pragma unroll
                for (int d = 16; d >= 1; d >>= 1) v = v + __shfl_xor(v, d);
                pv[p][r] = v / cdiv;
            }
        }
        if (a.vmode == 2) {
            final_norm(pv, hv);
        } else {
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int r = 0; r < 16; r++) hv[p][r] = pv[p][r];
        }
        barrier();   // every wave has finished reading the normalised streams
#pragma unroll
        for (int p = 0; p < NP; p++) publish(p, hv[p]);
        barrier();
        heads.pooled();
    }
    if constexpr (PROF) {
        BF_PHASE(PH_STORE);
        ph[PH_SYNC] = t_sync;
        ph[PH_TOTAL] = __builtin_readcyclecounter() - t_begin;
        if (lane == 0 && a.profile)
#pragma unroll
            for (int i = 0; i < N_PHASES; i++) atomicAdd(&a.profile[i], ph[i]);
    }
#undef BF_PHASE
}

template <int MODE, bool FP8, bool PROF = false, int NPOS = 2>
__global__ __launch_bounds__(512, 1) void duo_kernel(const KArgs a) {
    evaluate<MODE, FP8, PROF, NPOS>(a, (int)blockIdx.x, (int)gridDim.x);
}

// Both forms in one launch: a.pairs workgroups of two positions, and behind them those of one position that carry the last
// round.  As a launch of its own the last round waited until every pair was done, and over a leaf list (whose count is on
// the device, so that either may have nothing to do) it cost a launch: 577 positions 286.3 -> 283.6 us, 600 285.9 -> 283.0, e4m3, 600
// positions 372.1 -> 368.9, a list of 370 of 1000 with its expansion 183.9 -> 182.5; 700 and 2200 positions as before.  Over a list
// there is a workgroup for every pair of the buffer, and those without one only read the count (some 80 live of 4000, with compaction and expansion, 129.1 us, 120 of 12000 135.6).
template <int MODE, bool FP8>
__global__ __launch_bounds__(512, 1) void ragged_kernel(const KArgs a) {
    const int block = (int)blockIdx.x;
    if (block < a.pairs) evaluate<MODE, FP8, false, 2>(a, block, a.pairs);
    else evaluate<MODE, FP8, false, 1>(a, block - a.pairs, (int)gridDim.x - a.pairs);
}

// One launch of `kernel`; `lds_set`: the devices on which its dynamic LDS has been asked for (more than 64 KiB has to be, once
// per kernel and device)
inline hipError_t launch_kernel(void (*kernel)(KArgs), std::atomic<unsigned long long>& lds_set, int lds_bytes, int grid, const KArgs& k, hipStream_t stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipErrorInvalidDevice;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
    if (!(lds_set.load(std::memory_order_relaxed) & bit)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        if (e != hipSuccess) return e;
        lds_set.fetch_or(bit, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), lds_bytes, stream, k);
    return hipGetLastError();
}

template <int MODE, bool FP8 = false, bool PROF = false, int NPOS = 2>
hipError_t launch_duo(const KArgs& k, hipStream_t stream) {
    static std::atomic<unsigned long long> lds_set{0};
    return launch_kernel(&duo_kernel<MODE, FP8, PROF, NPOS>, lds_set, Cfg<FP8, NPOS>::LDS_BYTES, (k.n + NPOS - 1) / NPOS, k, stream);
}

// k.pairs workgroups of two positions and k.grid of one
template <int MODE, bool FP8>
hipError_t launch_ragged(const KArgs& k, hipStream_t stream) {
    static std::atomic<unsigned long long> lds_set{0};
    static_assert(Cfg<FP8, 2>::LDS_BYTES >= Cfg<FP8, 1>::LDS_BYTES, "both forms");
    return launch_kernel(&ragged_kernel<MODE, FP8>, lds_set, Cfg<FP8, 2>::LDS_BYTES, k.pairs + k.grid, k, stream);
}

}  // namespace duo
}  // namespace bf
