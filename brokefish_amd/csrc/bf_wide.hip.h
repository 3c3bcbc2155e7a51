// The 512-wide evaluator with TWO positions per workgroup of eight wavefronts.
//
// The decomposition is the eight-wavefront form of bf_board.hip.h (wavefront (q, sub) owns tiles 4q + 2sub and the next of
// the model width, which are also its two attention heads, and its half of quarter q's tiles in every matmul, and
// reads its blocks out of the quarter's weight stream where they lie), but every wavefront does its share for two
// positions, as in bf_duo.hip.h, so that a weight fragment out of L2 serves two positions.  With one position per
// workgroup the 50 MB of weights of every position cross a compute unit's path to L2, 60 % of that form's time.  The
// arithmetic is that of the other kernels operation for operation, and so are the bits.
//
// Two positions of this width fill a compute unit, so memory is shared over time:
//   registers  a wave's 64 of residual stream; during attention 48 of them lie in the hidden row's place in LDS
//   act / hid  the quantised rows of the width, 16 KiB a position, and three quarters of the hidden rows; the last
//              quarter takes the width's rows' place, which are dead by the time its scale is known
//   par        of a layer's side parameters what is needed when it is needed: LayerNorm 1; then biases and LayerNorm 2;
//              then the second feed-forward matmul's 128 * sum(w) where those were.  The first one's bias is read
//              from global memory.
// Every matmul of the width sums two k-chunks in float64: a tile's four products (chunk, position) have an accumulator each,
// and a position's epilogue runs under the product that follows its second chunk.
//
// What bounds it: a layer is 144,000 clocks of a SIMD, of which its two wavefronts' vector work is some 75,000 (the float64
// sums of two chunks alone 27,000: six instructions an element), fp32 matrix steps 16,500, int8 ones 50,000 less what runs
// under them, and fifteen exchanges some 15,000.  A call of 1500 positions: 4.38 ms with one position per workgroup, 3.40.  The 50 KB
// loop body matters (kernel alone, 3287 us): with every loop of a layer unrolled (95 KB, against 64 KiB of instruction cache for two compute
// units) and 50 registers spilled for it, 3776.  The weights' first touches are misses in every layer; sharing them out a
// phase ahead changed nothing (3327 against 3325).
//
// LDS map (bytes): [xch: 2 slots x 2 positions x 8 waves x 64 floats] [act: 16 KiB per position] [hid: 48 KiB per
// position] [tok: the activation scales of the rows that feed QKV, chunk by position by token] [key: what masks every
// token's scores as a key] [par: 1488 floats per quarter].  During the heads the normalised streams (64 KiB a position,
// fp32) take act and hid.
#pragma once

#include "bf_heads.hip.h"

namespace bf {
namespace wide {

using board::block_at;
using board::BlockAt;
using board::frag_mma;
using board::lds;
using board::lds_barrier;
using board::wait_vm;

struct Cfg : Layout<512> {
    static constexpr int NP = 2, NW = 8;
    static constexpr int XS = NP * NW * 64;               // floats of one exchange slot
    static constexpr int XCH_OFF = 0;
    static constexpr int ACT_OFF = XCH_OFF + 2 * XS * 4;
    static constexpr int ACT_P = NT * FRAG;               // a position's quantised row of the width
    static constexpr int HID_OFF = ACT_OFF + NP * ACT_P;
    static constexpr int HID_FRAGS = F / 32 - NT;         // tiles of the hidden row that lie in hid; the last NT lie in act
    static constexpr int HID_P = HID_FRAGS * FRAG;
    static constexpr int TOK_OFF = HID_OFF + NP * HID_P;
    static constexpr int KEY_OFF = TOK_OFF + KC * NP * 32 * 4;
    static constexpr int PAR_OFF = KEY_OFF + NP * 32 * 4;
    // a quarter's side parameters, in floats: [LayerNorm 1] [biases and scales of the attention phase, LayerNorm 2 -- or
    // 128 * sum(w)] [bias and scales of the feed-forward phase]
    static constexpr int P_LN1 = 0, P_ATT = 2 * CW, P_LN2 = P_ATT + (A_FLOATS - 2 * CW), P_WSUM = P_ATT, P_FFN = P_WSUM + KCF * CW,
                         PQ = P_FFN + (B_LDS_FLOATS - 2 * CW) + 48;
    static constexpr int LDS_BYTES = PAR_OFF + 4 * PQ * 4;
    static_assert(P_LN2 + 2 * CW <= P_FFN && LDS_BYTES <= 160 * 1024, "LDS budget: one workgroup per compute unit");
    static_assert(NT * 4 * FRAG * NP == NP * (ACT_P + HID_P), "normalised streams overlay");
    static_assert(NW * 48 * 256 == NP * HID_P, "parked registers overlay");
};

// The block numbers the kernel computes phase by phase, against block_at
template <int K_OUT, int K_FF1, int K_FF2, int NB>
constexpr bool block_at_agrees() {
    typedef Cfg C;
    for (int n = 0; n < NB; n++) {
        const BlockAt at = block_at<C::KC, C::TW, 2, true>(n);
        for (int sub = 0; sub < 2; sub++) {
            int w = 0;
            if (n < K_OUT) w = 12 * sub + n;
            else if (n < K_FF1) w = 24 + 4 * sub + (n - K_OUT);
            else if (n < K_FF2) w = 32 + 16 * ((n - K_FF1) / 4) + 4 * sub + (n - K_FF1) % 4;
            else w = 40 + 16 * ((n - K_FF2) % 8 / 2) + 4 * ((n - K_FF2) % 2) + 2 * sub + (n - K_FF2) / 8;
            if (at.a + sub * at.b != w) return false;
        }
    }
    return true;
}

template <int MODE, bool PROF = false>
__global__ __launch_bounds__(512, 1) void wide_kernel(const KArgs a) {
    constexpr bool ENC = MODE == MODE_ENC;
    static_assert(MODE != MODE_TAPS, "the debug taps are the one-position form's");
    typedef Cfg C;
    constexpr int NP = C::NP, D = C::D, NT = C::NT, TW = C::TW, TWW = 2, CW = C::CW, KC = C::KC, KCF = C::KCF;
    constexpr int STEPS = C::STEPS, BPW = C::BPW, HB = C::HB;
    constexpr int NB = BPW / 2;      // weight blocks a wave consumes per layer
    constexpr int HT = 2;            // hidden tiles a wave computes per feed-forward step
    constexpr int XS = C::XS, PS = C::NW * 64;
    constexpr int K_OUT = 3 * KC * TWW, K_FF1 = K_OUT + KC * TWW, K_FF2 = K_FF1 + STEPS * HT * KC;   // first blocks
    static_assert(KC == 2 && K_FF2 + TWW * KCF == NB, "a wave's blocks of a layer");
    static_assert(block_at_agrees<K_OUT, K_FF1, K_FF2, NB>(), "the phases' block numbers are block_at's");

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = wave & 3, sub = wave >> 2;
    const int tile0 = TW * q + TWW * sub, t0 = TWW * sub;   // first tile of the width; within the quarter
    const int t = lane & 31, g = lane >> 5;

    // the positions of this workgroup: its two slots of the launch, or those entries of the compacted leaf list (flags
    // without a list go to the one-position form).  A slot without a position computes its neighbour's again and stores
    // nothing; a workgroup without any leaves before the first barrier.
    int bp[NP];
    bool live[NP];
    {
        int cnt = a.n;
        if (a.leaf_index) {
            cnt = *a.leaf_count < a.n ? *a.leaf_count : a.n;
            if (a.list_split) cnt -= round_rest(cnt);
        }
        bool any = false;
        int some = 0;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int j = NP * (int)blockIdx.x + p;
            int b = j;
            bool ok = j < cnt;
            if (a.leaf_index) {
                b = ok ? __builtin_amdgcn_readfirstlane(a.leaf_index[j]) : 0;
                ok = ok && (unsigned)b < (unsigned)a.n;
            }
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
            __builtin_amdgcn_sched_barrier(0);                            \
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

    // the lane's offsets as opaque values, LDS addresses made where they are used, and weights through a buffer
    // descriptor: see bf_duo.hip.h
    int lane16 = lane * 16, lane4 = lane * 4;
    asm volatile("" : "+v"(lane16));
    asm volatile("" : "+v"(lane4));
    float* const xch = reinterpret_cast<float*>(lds + C::XCH_OFF);
    const float* const xlane = reinterpret_cast<const float*>(lds + C::XCH_OFF + lane4);
    uint8_t* const hid = lds + C::HID_OFF;
    uint8_t* const act = lds + C::ACT_OFF;
    float* const tok = reinterpret_cast<float*>(lds + C::TOK_OFF);
    float* const par = reinterpret_cast<float*>(lds + C::PAR_OFF) + q * C::PQ;
    const bool par_owner = sub == 0;
    auto here = [&](int wave_part, int at) -> uint8_t* {
        asm volatile("" : "+s"(wave_part));
        return lds + wave_part + at;
    };
    auto here_f = [&](int wave_part, int at) -> float* { return reinterpret_cast<float*>(here(wave_part, at)); };
    const int par_q = q * C::PQ * 4, par_t = par_q + 32 * t0 * 4, par_s = par_q + t0 * 4;   // par: the quarter's, the wave's tiles', their scales
    const int xch_w = wave * 256, frag_w = tile0 * FRAG, park_w = wave * 12 * FRAG, hid_w = (4 * q + HT * sub) * FRAG;
    const uint8_t* const wsrc = a.wstream + ((size_t)q * ((size_t)a.n_layers * BPW + HB + 1) + (size_t)a.l0 * BPW) * BLOCK;   // uniform
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wsrc), 0, ((a.n_layers - a.l0) * BPW + HB + 1) * BLOCK, 0x00027000);
    const __amdgpu_buffer_rsrc_t pbuf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.fparams + (size_t)q * a.n_layers * C::PW_FLOATS), 0, a.n_layers * C::PW_FLOATS * 4, 0x00027000);
    const float* const gp = a.fparams + (size_t)4 * a.n_layers * C::PW_FLOATS;
    auto fetch_par = [&](int at, int to, int nfloats) {   // floats [at, at + nfloats) of the quarter's parameters to par[to]
        uint8_t* const d = reinterpret_cast<uint8_t*>(par + to);
        const int bytes = nfloats * 4, full = bytes / FRAG, rem = (bytes % FRAG) / 16;
#pragma unroll
        for (int i = 0; i <= full; i++)
            if (i < full || lane < rem)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(pbuf, (__attribute__((address_space(3))) void*)(d + i * FRAG), 16, lane16, at * 4 + i * FRAG, 0, 0);
    };
    auto fetch_ln1 = [&](int l) { fetch_par(l * C::PW_FLOATS, C::P_LN1, 2 * CW); };
    auto fetch_att = [&](int l) {   // and what the feed-forward phase keeps
        fetch_par(l * C::PW_FLOATS + 2 * CW, C::P_ATT, C::A_FLOATS - 2 * CW);
        fetch_par(l * C::PW_FLOATS + C::A_FLOATS, C::P_LN2, 2 * CW);
        fetch_par(l * C::PW_FLOATS + C::A_FLOATS + 2 * CW, C::P_FFN, C::B_LDS_FLOATS - 2 * CW);
    };
    auto fetch_wsum = [&](int l) { fetch_par(l * C::PW_FLOATS + C::A_FLOATS + C::B_WSUM, C::P_WSUM, KCF * CW); };
    // places in par; `at` as in part A and in part B of a layer's side parameters
    auto p_att = [&](int wave_part, int at) -> float* { return here_f(wave_part, C::PAR_OFF + (C::P_ATT - 2 * CW + at) * 4); };
    auto p_ffn = [&](int wave_part, int at) -> float* { return here_f(wave_part, C::PAR_OFF + (C::P_FFN - 2 * CW + at) * 4); };

    // The weight fragments in flight or in use: a block.  While the second position consumes fragment f of a block, fragment f
    // of the wave's next block takes its place.
    v4i frt[8];
    auto load_frag = [&](int block, int f) {
        frt[f] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf, lane16, block * BLOCK + f * FRAG, 0));
    };
    // where the wave's blocks of a layer lie in the quarter's stream (block_at, by phase)
    auto block_qkv = [&](int n) { return 3 * KC * TWW * sub + n; };
    auto block_out = [&](int n) { return 3 * KC * TW + KC * TWW * sub + n; };
    auto block_ff1 = [&](int st, int n) { return 4 * KC * TW + (4 * KC + 2 * TW) * st + KC * HT * sub + n; };
    auto block_ff2 = [&](int i, int cc) { return 4 * KC * TW + (4 * KC + 2 * TW) * (cc >> 1) + 4 * KC + (cc & 1) * TW + TWW * sub + i; };

    auto xsum2 = [&](const float (&part)[NP], int slot) -> float {
#pragma unroll
        for (int p = 0; p < NP; p++) here_f(xch_w, C::XCH_OFF + (slot * XS + p * PS) * 4)[lane] = part[p];
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
    auto xmax_put = [&](const float (&am)[NP], int at) { here_f(xch_w, C::XCH_OFF + at * 4)[lane] = Rows<NP>::max(am); };
    // AFTER() runs behind the first barrier
    auto layernorm2 = [&](const float (&x)[NP][TWW][16], const float* gamma, const float* beta, float (&y)[NP][TWW][16], auto&& after) {
        float part[NP], mean[NP], rstd[NP];
        auto tiles = [&](auto&& term) {
#pragma unroll
            for (int p = 0; p < NP; p++) {
                float ts[TWW];
#pragma unroll
                for (int i = 0; i < TWW; i++) {
                    float acc = 0.0f;
#pragma unroll
                    for (int r = 0; r < 16; r++) acc = term(p, i, r, acc);
                    ts[i] = acc;
                }
                part[p] = ts[0] + ts[1];
            }
        };
        tiles([&](int p, int i, int r, float acc) { return acc + x[p][i][r]; });
        Rows<NP>::each(xsum2(part, 0) * (1.0f / D), mean);
        after();
        tiles([&](int p, int i, int r, float acc) {
            const float d = x[p][i][r] - mean[p];
            return __builtin_fmaf(d, d, acc);
        });
        Rows<NP>::each(recip_sqrt(xsum2(part, 1) * (1.0f / D) + a.eps), rstd);
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f ga = ldg4(gamma + 32 * i + 8 * j + 4 * g);
                const v4f be = ldg4(beta + 32 * i + 8 * j + 4 * g);
#pragma unroll
                for (int p = 0; p < NP; p++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float d = x[p][i][4 * j + k] - mean[p];
                        y[p][i][4 * j + k] = __builtin_fmaf(d * rstd[p], ga[k], be[k]);
                    }
            }
    };
    // signed quantiser of both positions' rows: a scale per row and 256-wide chunk (quarters 0, 1 and 2, 3)
    auto quant_exchange2 = [&](const float (&y)[NP][TWW][16], float (&sa)[NP][KC], bool publish_scales, bool landed) {
        float am[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            am[p] = 0.0f;
#pragma unroll
            for (int i = 0; i < TWW; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) am[p] = __builtin_fmaxf(am[p], __builtin_fabsf(y[p][i][r]));
        }
        xmax_put(am, 0);
        barrier();
        float mw[8], sr[KC];
#pragma unroll
        for (int w = 0; w < C::NW; w++) mw[w] = xlane[w * 64];
#pragma unroll
        for (int c = 0; c < KC; c++) {
            sr[c] = row_scale<false>(vmax(vmax3(mw[2 * c], mw[2 * c + 1], mw[2 * c + 4]), mw[2 * c + 5]));
            float each[NP];
            Rows<NP>::each(sr[c], each);
#pragma unroll
            for (int p = 0; p < NP; p++) sa[p][c] = each[p];
            if (publish_scales && wave == 0) here_f(0, C::TOK_OFF + c * NP * 128)[lane] = sr[c];
        }
        const Quot br = quot_by(q < 2 ? sr[0] : sr[1]);
        float hi[NP], lo[NP];
        Rows<NP>::each(br.hi, hi);
        Rows<NP>::each(br.lo, lo);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const Quot by = {hi[p], lo[p]};
#pragma unroll
            for (int i = 0; i < TWW; i++) {
                v4i w;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    w[j] = (int)quant4<false>(y[p][i][4 * j], y[p][i][4 * j + 1], y[p][i][4 * j + 2], y[p][i][4 * j + 3], by);
                *reinterpret_cast<v4i*>(here(frag_w, C::ACT_OFF + p * C::ACT_P + i * FRAG) + lane16) = w;
            }
        }
        if (landed && par_owner) wait_vm<0>();   // the parameters asked for behind the first barrier
        barrier();
    };
    const uint8_t* const act0 = act + lane16;
    const uint8_t* const hid0 = hid + lane16;
    auto ldsfrag = [&](const uint8_t* p) -> v4i { return *reinterpret_cast<const v4i*>(p); };

    // ---- start the weight stream and the first layer's parameters --------------------------------
    if (nl_run > 0) {
#pragma unroll
        for (int f = 0; f < 8; f++) load_frag(block_qkv(0), f);
        if (par_owner) {
            fetch_ln1(a.l0);
            fetch_att(a.l0);
        }
    }

    // ---- embedding (this wave's tiles, both positions), or the caller's stream -----------------------------
    float x[NP][TWW][16];
    unsigned alive[NP];
    int ctrl[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int b = bp[p];
        const unsigned word = ENC ? (a.taps.alive[(size_t)b * T + t] ? 0u : 0x800u) : a.boards[(size_t)b * T + t];
        ctrl[p] = ENC ? 1 : a.control[b];
        alive[p] = (unsigned)__ballot(((word >> 11) & 1) == 0 && g == 0);
        if (wave == 0 && g == 0) reinterpret_cast<float*>(lds + C::KEY_OFF)[p * 32 + t] = ((word >> 11) & 1) == 0 ? 0.0f : -__builtin_inff();
        if (ENC) {
#pragma unroll
            for (int i = 0; i < TWW; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4f v = stream_in(a.taps, ((size_t)b * T + t) * D + 32 * (tile0 + i) + 8 * j + 4 * g);
#pragma unroll
                    for (int k = 0; k < 4; k++) x[p][i][4 * j + k] = v[k];
                }
        } else {
            const int stm = ctrl[p] < 0;
            int clock = (ctrl[p] < 0 ? -ctrl[p] : ctrl[p]) - 1;
            clock = clock < 0 ? 0 : (clock > 100 ? 100 : clock);
            int rp = a.rep[b];
            rp = rp > 2 ? 2 : rp;
            int ts = ((word >> 6) & 7) * 2 + ((word >> 9) & 1);
            ts = ts > 11 ? 11 : ts;
            const int ct = ((word >> 10) & 1) * 2 + stm;
            const int own = 32 * tile0 + 4 * g;
            const float* e_sq = gp + C::G_SQ + (word & 63) * D + own;
            const float* e_ts = gp + C::G_TS + ts * D + own;
            const float* e_ct = gp + C::G_CT + ct * D + own;
            const float* e_ck = gp + C::G_CLOCK + clock * D + own;
            const float* e_rp = gp + C::G_REP + rp * D + own;
#pragma unroll
            for (int i = 0; i < TWW; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int c = 32 * i + 8 * j;
                    const v4f vs = ldg4(e_sq + c), vt = ldg4(e_ts + c), vc = ldg4(e_ct + c);
                    const v4f vk = ldg4(e_ck + c), vr = ldg4(e_rp + c);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float per_board = vk[k] + vr[k];
                        float v = vs[k] + vt[k];
                        v = v + vc[k];
                        x[p][i][4 * j + k] = v + per_board;
                    }
                }
        }
    }
    wait_vm<0>();   // the parameters have landed (published to the quarter's other wave by the next barrier)
    BF_PHASE(PH_EMBED);

    const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    auto none = [](int) {};
    auto nothing = []() {};
    for (int l = a.l0; l < a.l1; l++) {
        const int li = l - a.l0;
        const int lnext = l + 1 < a.l1 ? l + 1 : l;   // after the last layer the same layer is fetched again (and never used)
        const int lbase = li * BPW, lfollow = (lnext - a.l0) * BPW;
        // One product of position p with the block in frt: eight 32-deep steps against the operand row at BSRC, each
        // fragment fetched from LDS one step ahead; the second position replaces each fragment by block NEXT's.
        // BETWEEN(s) runs after step s has been issued: an eighth of an earlier epilogue.
#define BF_WIDE_CHAIN(SWAP, p, BSRC, NEXT, INIT, R, BETWEEN)                                         \
    do {                                                                                             \
        const uint8_t* const b_ = (BSRC);                                                            \
        v4i op_[2];                                                                                  \
        op_[0] = ldsfrag(b_);                                                                        \
        (R) = (INIT);                                                                                \
        _Pragma("unroll") for (int s_ = 0; s_ < 8; s_++) {                                           \
            if (s_ + 1 < 8) op_[(s_ + 1) & 1] = ldsfrag(b_ + (s_ + 1) * FRAG);                       \
            (R) = frag_mma<SWAP>(frt[s_], op_[s_ & 1], (R));                                         \
            BETWEEN(s_);                                                                             \
            __builtin_amdgcn_sched_barrier(0);                                                       \
            if ((p) == 1) load_frag(NEXT, s_);                                                       \
        }                                                                                            \
    } while (0)
        // A tile's four products: chunk 0 of both positions (B1 and B2 under them), chunk 1 of both (B4 under the second one:
        // position 0's epilogue; position 1's is the caller's, behind them or as the next tile's B1).  The tile's second block is
        // BLK + 1, the one behind it NEXT.
        v16i acc[NP][KC];
#define BF_WIDE_TILE(SWAP, BLK, NEXT, B1, B2, B4)                                                    \
    do {                                                                                             \
        BF_WIDE_CHAIN(SWAP, 0, act0, 0, zero, acc[0][0], B1);                                        \
        BF_WIDE_CHAIN(SWAP, 1, act0 + C::ACT_P, (BLK) + 1, zero, acc[1][0], B2);                     \
        BF_WIDE_CHAIN(SWAP, 0, act0 + 8 * FRAG, 0, zero, acc[0][1], none);                           \
        BF_WIDE_CHAIN(SWAP, 1, act0 + C::ACT_P + 8 * FRAG, NEXT, zero, acc[1][1], B4);               \
    } while (0)
        // element e of position p's tile: the chunks' accumulators times their scales, summed in float64, cast once
        auto sum2 = [&](int p, int e, float s0, float s1) -> float {
            return (float)__builtin_fma((double)acc[p][1][e], (double)s1, (double)acc[p][0][e] * (double)s0);
        };

        // ---- LayerNorm 1, quantise, exchange -----------------------------------------------------------
        float sa[NP][KC];
        {
            float y[NP][TWW][16];
            auto after = [&]() {   // both waves of the quarter are through with the last layer's parameters
                if (par_owner && li > 0) fetch_att(l);
            };
            layernorm2(x, here_f(par_t, C::PAR_OFF + C::P_LN1 * 4), here_f(par_t, C::PAR_OFF + (C::P_LN1 + CW) * 4), y, after);
            quant_exchange2(y, sa, true, true);
        }
        // three quarters of the residual stream wait in the hidden rows' place
        auto each_parked = [&](auto&& f) {
#pragma unroll
            for (int n = 1; n < 4; n++)
#pragma unroll
                for (int j = 0; j < 4; j++) f(n >> 1, n & 1, j, (n - 1) * 4 + j);
        };
        {
            uint8_t* const to = here(park_w, C::HID_OFF) + lane16;
            each_parked([&](int p, int i, int j, int at) {
                *reinterpret_cast<v4f*>(to + at * FRAG) = v4f{x[p][i][4 * j], x[p][i][4 * j + 1], x[p][i][4 * j + 2], x[p][i][4 * j + 3]};
            });
        }
        BF_PHASE(PH_LN1);

        // ---- attention: this wave's two heads, both positions ---------------------------------------------
        // The loops of a layer stay loops (heads, feed-forward steps, chunks): unrolled, a layer is 95 KiB of code, and two compute
        // units share 64 KiB of instruction cache.
        float o[NP][TWW][16] = {};
#pragma unroll
        for (int i = 0; i < TWW; i++) {
            const int blk = lbase + block_qkv(3 * KC * i), behind = i + 1 < TWW ? blk + 3 * KC : lbase + block_out(0);
            float qf[NP][16], kf[NP][16], vf[NP][16];
            if (sub) __builtin_amdgcn_s_setprio(2);   // the SIMD's younger wavefront first, see bf_duo.hip.h (3325 -> 3287 us)
            v4f bias[4];
            const float sw = *p_att(par_s + i * 4, C::A_SW);
            load_tile16(p_att(par_t + 128 * i, C::A_BQ), g, bias);
            auto epi_q = [&](int p, int s) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) qf[p][e] = sum2(p, e, sa[p][0], sa[p][1]) * sw + bias[e / 4][e % 4];
            };
            auto q0 = [&](int s) { epi_q(0, s); };
            auto q1 = [&](int s) { epi_q(1, s); };
            BF_WIDE_TILE(false, blk, blk + 2, none, none, q0);
            v4f biask[4];
            const float swk = *p_att(par_s + i * 4, C::A_SW + TW);
            auto epi_k = [&](int p, int s) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) kf[p][e] = sum2(p, e, sa[p][0], sa[p][1]) * swk + biask[e / 4][e % 4];
            };
            auto load_k = [&](int s) { if (s == 0) load_tile16(p_att(par_t + 128 * i, C::A_BK), g, biask); };
            auto k0 = [&](int s) { epi_k(0, s); };
            BF_WIDE_TILE(false, blk + 2, blk + 4, q1, load_k, k0);
#pragma unroll
            for (int s = 0; s < 8; s++) epi_k(1, s);
            __builtin_amdgcn_s_setprio(0);
            // scores, transposed: lane = query token, register r = key ch(r, g)
            float pr[NP][16], rl[NP];
#pragma unroll
            for (int p = 0; p < NP; p++) {
                v16f sc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < 16; r++) sc = BF_F32MMA(kf[p][r], qf[p][r], sc);
#pragma unroll
                for (int r = 0; r < 16; r++) pr[p][r] = sc[r];
                pin16(pr[p]);
            }
            BF_PHASE(PH_QKV);
#pragma unroll
            for (int p = 0; p < NP; p++) {
                float mx = -__builtin_inff();
                v4f kb[4];
                load_tile16(here_f(0, C::KEY_OFF + p * 128), g, kb);
#pragma unroll
                for (int r = 0; r < 16; r++) {   // scaled and masked in one operation (see bf_duo.hip.h)
                    pr[p][r] = __builtin_fmaf(pr[p][r], 0.17677669529663687f, kb[r / 4][r % 4]);
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
                pin16(pr[p]);
            }
            // V: rows are tokens, so the activation scales are those of token ch(e, g)
            const float swv = *p_att(par_s + i * 4, C::A_SW + 2 * TW);
            const float bv = p_att(par_t + 128 * i, C::A_BV)[t];
            auto epi_v = [&](int p, int s) {
                const int e = 2 * s;
                const v2f s0 = *reinterpret_cast<const v2f*>(here_f(0, C::TOK_OFF + (p * 32 + 8 * (e / 4) + e % 4) * 4) + 4 * g);
                const v2f s1 = *reinterpret_cast<const v2f*>(here_f(0, C::TOK_OFF + (NP * 32 + p * 32 + 8 * (e / 4) + e % 4) * 4) + 4 * g);
#pragma unroll
                for (int u = 0; u < 2; u++) vf[p][e + u] = sum2(p, e + u, s0[u], s1[u]) * swv + bv;
            };
            auto v0 = [&](int s) { epi_v(0, s); };
            BF_WIDE_TILE(true, blk + 4, behind, none, none, v0);
#pragma unroll
            for (int s = 0; s < 8; s++) epi_v(1, s);
#pragma unroll
            for (int p = 0; p < NP; p++) {
                v16f oa = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < 16; r++) oa = BF_F32MMA(vf[p][r], pr[p][r] * rl[p], oa);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    o[p][0][r] = o[p][1][r];
                    o[p][1][r] = oa[r];
                }
                pin16(o[p][1]);
            }
            BF_PHASE(PH_ATTN);
        }

        // ---- output projection + residual ------------------------------------------------------------------
        {
            float so[NP][KC];
            quant_exchange2(o, so, false, false);
            {
                const uint8_t* const from = here(park_w, C::HID_OFF) + lane16;
                each_parked([&](int p, int i, int j, int at) {
                    const v4f v = *reinterpret_cast<const v4f*>(from + at * FRAG);
#pragma unroll
                    for (int k = 0; k < 4; k++) x[p][i][4 * j + k] = v[k];
                });
            }
            v4f bo[TWW][4];
            float sw[TWW];
            auto epi_o = [&](int i, int p, int s) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) x[p][i][e] = x[p][i][e] + (sum2(p, e, so[p][0], so[p][1]) * sw[i] + bo[i][e / 4][e % 4]);
            };
#pragma unroll
            for (int i = 0; i < TWW; i++) {
                sw[i] = *p_att(par_s, C::A_SW + 3 * TW + i);
                auto before = [&](int s) { if (i > 0) epi_o(i - 1, 1, s); };
                auto load_b = [&](int s) { if (s == 0) load_tile16(p_att(par_t, C::A_BOUT + 32 * i), g, bo[i]); };
                auto first = [&](int s) { epi_o(i, 0, s); };
                BF_WIDE_TILE(false, lbase + block_out(KC * i), lbase + (i + 1 < TWW ? block_out(KC * (i + 1)) : block_ff1(0, 0)), before, load_b, first);
            }
#pragma unroll
            for (int s = 0; s < 8; s++) epi_o(TWW - 1, 1, s);
        }
        BF_PHASE(PH_OUT);

        // ---- feed-forward ---------------------------------------------------------------------------------
        {
            float y[NP][TWW][16];
            layernorm2(x, here_f(par_t, C::PAR_OFF + C::P_LN2 * 4), here_f(par_t, C::PAR_OFF + (C::P_LN2 + CW) * 4), y, nothing);
            quant_exchange2(y, sa, false, false);
        }
        if (par_owner) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            fetch_wsum(l);
            fetch_ln1(lnext);
        }
        BF_PHASE(PH_LN2);
        // First matmul, step by step: each step's two 256-wide chunks are quantised as soon as the step is complete.  The last
        // step's tiles go where the width's rows were: every wave has read them when it has published its maximum.
        float sh[KCF] = {};   // the chunks' scales, position 0's in the lower lanes, position 1's in the upper ones
#pragma unroll 1
        for (int st = 0; st < STEPS; st++) {
            const int blk = lbase + block_ff1(st, 0), behind = lbase + (st + 1 < STEPS ? block_ff1(st + 1, 0) : block_ff2(0, 0));
            float hf[NP][HT][16];
            float am[NP] = {0.0f, 0.0f};
            v4f b1[HT][4];
            float sw1[HT];
            auto epi_f = [&](int i, int p, int s) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) {
                    // the ReLU is in the hidden quantiser's saturation, and the running maximum starts at 0
                    const float v = sum2(p, e, sa[p][0], sa[p][1]) * sw1[i] + b1[i][e / 4][e % 4];
                    hf[p][i][e] = v;
                    am[p] = __builtin_fmaxf(am[p], v);
                }
            };
#pragma unroll
            for (int i = 0; i < HT; i++) {
                sw1[i] = *p_ffn(par_s + 16 * st, C::B_SW + i);
                auto before = [&](int s) { if (i > 0) epi_f(i - 1, 1, s); };
                auto load_b = [&](int s) {
                    if (s == 0)
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            b1[i][j] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                pbuf, 16 * g, (l * C::PW_FLOATS + C::A_FLOATS + C::B_BFF1 + 128 * st + 32 * (HT * sub + i) + 8 * j) * 4, 0));
                };
                auto first = [&](int s) { if (i + 1 < HT) epi_f(i, 0, s); };
                BF_WIDE_TILE(false, blk + KC * i, i + 1 < HT ? blk + KC * (i + 1) : behind, before, load_b, first);
            }
#pragma unroll
            for (int s = 0; s < 8; s++) epi_f(HT - 1, 0, s);
#pragma unroll
            for (int s = 0; s < 8; s++) epi_f(HT - 1, 1, s);
            // the maxima of consecutive steps go through different exchange slots (1, whose last use was a LayerNorm sum two
            // barriers ago, then 0)
            const int xs = (st & 1) ? 0 : XS;
            here_f(xch_w + xs * 4, C::XCH_OFF)[lane] = Rows<NP>::max(am);
            barrier();
            float hi[NP], lo[NP];
            {
                float mw[8];
#pragma unroll
                for (int w = 0; w < C::NW; w++) mw[w] = (xlane + xs)[w * 64];
#pragma unroll
                for (int c = 0; c + 2 < KCF; c++) sh[c] = sh[c + 2];   // in order when the last step is done
#pragma unroll
                for (int c = 0; c < 2; c++)
                    sh[KCF - 2 + c] = hidden_scale<false>(vmax(vmax3(mw[2 * c], mw[2 * c + 1], mw[2 * c + 4]), mw[2 * c + 5]));
                const Quot br = quot_by(q < 2 ? sh[KCF - 2] : sh[KCF - 1]);
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
                    for (int j = 0; j < 4; j++)
                        w[j] = (int)(quant4_relu_u8(hf[p][i][4 * j], hf[p][i][4 * j + 1], hf[p][i][4 * j + 2], hf[p][i][4 * j + 3], by) ^ 0x80808080u);
                    const int to = st + 1 < STEPS ? C::HID_OFF + p * C::HID_P + 16 * st * FRAG : C::ACT_OFF + p * C::ACT_P;
                    *reinterpret_cast<v4i*>(here(hid_w + to, i * FRAG) + lane16) = w;
                }
            }
        }
        barrier();   // the whole hidden rows of both positions are in LDS
        BF_PHASE(PH_FF1);
        // Second matmul: an output tile over the KCF k-chunks in turn; the accumulator starts at 128 * sum(w), the offset of the
        // unsigned bytes stored as q - 128; the sums over the chunks are float64.
#pragma unroll 1
        for (int i = 0; i < TWW; i++) {
            double o64[NP][16] = {};
            v16i ac[2] = {zero, zero};
            double by[NP] = {0.0, 0.0};      // the scales of the chunk whose accumulators wait for their epilogue
            auto epi_2 = [&](int p, int s) {
#pragma unroll
                for (int e = 2 * s; e < 2 * s + 2; e++) o64[p][e] = __builtin_fma((double)ac[p][e], by[p], o64[p][e]);
            };
            auto epi_20 = [&](int s) { epi_2(0, s); };
            auto epi_21 = [&](int s) { epi_2(1, s); };
#pragma unroll 1
            for (int cc = 0; cc < KCF; cc++) {
                v16i init;
                {
                    v4i w0[4];
                    load_tile16i(here_f(par_t + (cc * CW + 32 * i) * 4, C::PAR_OFF + C::P_WSUM * 4), g, w0);
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int k = 0; k < 4; k++) init[4 * j + k] = w0[j][k];
                }
                float sc[NP];
                const float first = sh[0];
                Rows<NP>::each(first, sc);
#pragma unroll
                for (int c = 0; c < KCF; c++) sh[c] = c + 1 < KCF ? sh[c + 1] : first;
                const bool in_hid = cc < C::HID_FRAGS / 8;
                const uint8_t* const row = lds + lane16 + (in_hid ? C::HID_OFF + 8 * cc * FRAG : C::ACT_OFF + (8 * cc - C::HID_FRAGS) * FRAG);
                const int next = cc + 1 < KCF ? lbase + block_ff2(i, cc + 1) : i + 1 < TWW ? lbase + block_ff2(i + 1, 0) : lfollow + block_qkv(0);
                BF_WIDE_CHAIN(false, 0, row, 0, init, ac[0], epi_21);
                by[0] = (double)sc[0];
                by[1] = (double)sc[1];
                BF_WIDE_CHAIN(false, 1, row + (in_hid ? C::HID_P : C::ACT_P), next, init, ac[1], epi_20);
            }
#pragma unroll
            for (int s = 0; s < 8; s++) epi_21(s);
            v4f b2[4];
            load_tile16(p_ffn(par_t + 32 * i * 4, C::B_BFF2), g, b2);
            const float sw = *p_ffn(par_s + i * 4, C::B_SW + 16);
            // tile i is in front: the two change places, and are back when both are done
#pragma unroll
            for (int p = 0; p < NP; p++) {
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const float done = x[p][0][e] + ((float)o64[p][e] * sw + b2[e / 4][e % 4]);
                    x[p][0][e] = x[p][1][e];
                    x[p][1][e] = done;
                }
                pin16(x[p][0]);
                pin16(x[p][1]);
            }
        }
        BF_PHASE(PH_FF2);
#undef BF_WIDE_TILE
#undef BF_WIDE_CHAIN
    }
    if constexpr (ENC) {
#pragma unroll
        for (int p = 0; p < NP; p++)
            if (live[p])
#pragma unroll
                for (int i = 0; i < TWW; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        stream_out(a.taps, ((size_t)bp[p] * T + t) * D + 32 * (tile0 + i) + 8 * j + 4 * g,
                                   v4f{x[p][i][4 * j], x[p][i][4 * j + 1], x[p][i][4 * j + 2], x[p][i][4 * j + 3]});
        return;
    }

    // ---- final norm and heads --------------------------------------------------------------------------
    constexpr int STREAM_P = NT * 4 * FRAG;   // a position's normalised stream, bytes: both take act and hid
    Heads<NP, HB, 8> heads(a, BPW, lane, wave, bp, live, ctrl, C::ACT_OFF, STREAM_P);
    heads.ask();
    float hn[NP][TWW][16];
    layernorm2(x, gp + C::G_NFG + 32 * tile0, gp + C::G_NFB + 32 * tile0, hn, nothing);   // its barriers: every wave is done with the hidden rows
    auto publish = [&](const float (&v)[NP][TWW][16]) {
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int i = 0; i < TWW; i++) heads.publish(p, tile0 + i, v[p][i]);
    };
    publish(hn);
    barrier();
    heads.products();
    BF_PHASE(PH_HEADS);
    heads.store(tok, barrier);   // where the activation scales were
    // ---- pooled value heads (see bf_duo.hip.h) ----------------------------------------------------------
    if (a.vmode != 0) {
        float pv[NP][TWW][16], hv[NP][TWW][16];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const bool lv = (alive[p] >> t) & 1u;
            const float cdiv = (float)(__builtin_popcount(alive[p]) > 0 ? __builtin_popcount(alive[p]) : 1);
#pragma unroll
            for (int i = 0; i < TWW; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float v = lv ? (a.vmode == 1 ? hn[p][i][r] : x[p][i][r]) : 0.0f;
#pragma unroll
                    for (int d = 16; d >= 1; d >>= 1) v = v + __shfl_xor(v, d);
                    pv[p][i][r] = v / cdiv;
                }
        }
        if (a.vmode == 2) {
            layernorm2(pv, gp + C::G_NFG + 32 * tile0, gp + C::G_NFB + 32 * tile0, hv, nothing);
        } else {
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int i = 0; i < TWW; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) hv[p][i][r] = pv[p][i][r];
        }
        barrier();   // every wave has finished reading the normalised streams
        publish(hv);
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

template <int MODE, bool PROF = false>
hipError_t launch_wide(const KArgs& k, hipStream_t stream) {
    // more than 64 KiB of dynamic LDS has to be requested once per kernel and device
    static std::atomic<unsigned long long> lds_set{0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipErrorInvalidDevice;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
    if (!(lds_set.load(std::memory_order_relaxed) & bit)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&wide_kernel<MODE, PROF>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
        if (e != hipSuccess) return e;
        lds_set.fetch_or(bit, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL((wide_kernel<MODE, PROF>), dim3((k.n + 1) / 2), dim3(512), Cfg::LDS_BYTES, stream, k);
    return hipGetLastError();
}

}  // namespace wide
}  // namespace bf
