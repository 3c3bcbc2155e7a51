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
// So a layer has two exchanges, its weights are read once per team except the output projection's, and a wavefront
// never has more than one tile (width 512: two) in a matmul.  Measured: one position 124 -> 90 us, 64 positions
// 120 -> 95, e4m3 155 -> 106; width 512, 16 layers: one position 750 -> 346 us, 32 positions 727 -> 381.  The arithmetic is that of the other kernels,
// operation for operation: the results are bit-identical to theirs.
//
// An exchange: a wavefront stores its piece, waits until the L2 has it (vmcnt), and stores a flag; the wavefronts that
// need the piece poll the flag past their L1 (sc1) and then load the piece past it (dword flags; polling tags inside
// the data itself was slower, every poll is 16 KiB).  Members sit behind one L2
// because workgroups go to the XCDs in turn (blockIdx % 8; bf_team_setup looks at the device before the form is
// used).  Measured on its own: 3.0 k clocks from store to data with 4 x 32 KiB exchanged.  Flags count layers over
// all launches of a workspace (each member keeps the count, a multiple it adds at its end), so nothing is
// cleared between launches.  Waiting is bounded: a wavefront that has waited some seconds gives up, publishes nothing
// any more and makes its part of the stream NaN.  Members of a team are consecutive workgroups of their XCD and
// are dispatched in order, so at most NWG - 1 workgroups of a launch per XCD ever wait for a unit to come free.
//
// No exchange buffer is written twice in a layer, and one set per team is enough: a member writes A or B of
// layer l + 1 only after barriers that follow its wavefronts' loads of B of layer l from all members, and every
// wavefront loads A of a layer before it stores its B.
//
// LDS map: [xch: 3 slots x 8 waves x 64 floats] [act: the quantised row of the width] [hid: the quantised chunk]
// [tok: activation scales of the row that feeds QKV] [qkv: Q, K, V of two heads, 24 KiB] [par: a layer's side
// parameters, twice].  During the heads the normalised stream (fp32) overlays qkv / par.
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
    static constexpr int TWW = L::NT / NW;          // tiles of the width a wavefront owns
    static constexpr int NHW = L::NT / NWG;         // heads of a member
    static_assert(NHW == 2, "two heads per member");
    static constexpr int XS = NW * 64;
    static constexpr int XCH_OFF = 0;
    static constexpr int ACT_OFF = XCH_OFF + 3 * XS * 4;
    static constexpr int HID_OFF = ACT_OFF + L::NT * FRAG;
    static constexpr int TOK_OFF = HID_OFF + 8 * FRAG;
    static constexpr int QKV_OFF = TOK_OFF + FRAG;
    static constexpr int PAR_OFF = QKV_OFF + NHW * 3 * 4 * FRAG;
    static constexpr int PAR_BYTES = 4 * L::PW_FLOATS * 4;
    static constexpr int USED_BYTES = PAR_OFF + 2 * PAR_BYTES;
    // more than half a compute unit's LDS: never two workgroups on one unit while another is empty
    static constexpr int LDS_BYTES = USED_BYTES < 81 * 1024 ? 81 * 1024 : USED_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
    static_assert(QKV_OFF + L::NT * 4 * FRAG <= LDS_BYTES, "normalised stream overlay");
    // a team's part of the workspace, bytes
    static constexpr int FLAG_A = 64, FLAG_B = 128;           // dwords: first flag of exchange A, of exchange B
    static constexpr int WS_A = 4096;                         // [tile][quad 4][64 lanes] 16 bytes
    static constexpr int WS_B = WS_A + L::NT * 4 * FRAG;      // [member][wave][4 TWW quads + scale][64 lanes] 16 bytes
    static constexpr int B_PIECE = (4 * TWW + 1) * FRAG;
    static constexpr int WS_BYTES = WS_B + NWG * NW * B_PIECE;
    static_assert(NWG <= FLAG_A && FLAG_A + 2 * L::NT <= FLAG_B && (FLAG_B + NWG * NW) * 4 <= WS_A, "flags");
};

constexpr int SPIN_LIMIT = 1 << 23;   // polls of some 600 clocks: about two seconds
constexpr int SC1 = 16;               // cache policy of a load that goes past the L1

// the other of lanes l and l ^ 16, and both in row order
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
    constexpr int BPW = C::BPW, HB = C::HB, XS = C::XS;
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
    int* const flags = reinterpret_cast<int*>(ws);
    const int tag0 = __builtin_amdgcn_readfirstlane(flags[m]);   // layers of the launches before this one
    bool dead = false;                                           // this wave has given up waiting

    float* const xch = reinterpret_cast<float*>(lds + C::XCH_OFF);
    uint8_t* const act = lds + C::ACT_OFF;
    uint8_t* const hid = lds + C::HID_OFF;
    float* const tok = reinterpret_cast<float*>(lds + C::TOK_OFF);
    float* const qkv = reinterpret_cast<float*>(lds + C::QKV_OFF);
    const float* const gp = a.fparams + (size_t)4 * a.n_layers * C::PW_FLOATS;
    auto par = [&](int l, int quarter) { return reinterpret_cast<const float*>(lds + C::PAR_OFF + (l & 1) * C::PAR_BYTES) + quarter * C::PW_FLOATS; };
    auto fetch_par = [&](int l) {   // a quarter's part A by its first wave, part B by its second
        const float* src = a.fparams + ((size_t)q * a.n_layers + l) * C::PW_FLOATS;
        float* dst = const_cast<float*>(par(l, q));
        if (wave & 1) dma(src + C::A_FLOATS, dst + C::A_FLOATS, C::B_FLOATS, lane);
        else dma(src, dst, C::A_FLOATS, lane);
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
    // Two register sets of KC blocks: SA serves QKV, (width 512) the second tile of the output projection, and
    // the second feed-forward matmul; SB the output projection and the first.  A set is filled as soon as it is
    // free, a LayerNorm, an attention or an exchange ahead of its use.
    v4i SA[KC][8], SB[KC][8];
    const int hh = wave & 1, tq = wave >> 1;        // QKV: waves 0..5 take tile tq (Q, K, V) of head hh
    const int head = 2 * m + hh, hq = head / TW, hi = head % TW;
    auto fetch_qkv = [&](int l) {
        if (tq < 3) {
#pragma unroll
            for (int c = 0; c < KC; c++) load_block(SA[c], hq, l, 3 * KC * hi + tq * KC + c);
        } else {   // nothing: the set's old contents end here, or they would stay in registers up to this point
#pragma unroll
            for (int c = 0; c < KC; c++)
#pragma unroll
                for (int s = 0; s < 8; s++) asm volatile("" : "=v"(SA[c][s]));
        }
    };
    auto fetch_out = [&](v4i (&w)[KC][8], int l, int i) {
#pragma unroll
        for (int c = 0; c < KC; c++) load_block(w[c], q, l, 3 * KC * TW + KC * (iq0 + i) + c);
    };
    const int fq = 2 * (m & 1) + (wave >> 2), fh = wave & 3, fst = m >> 1;   // hidden tile 8 m + wave: its quarter, number there, step
    auto fetch_ff1 = [&](int l) {
#pragma unroll
        for (int c = 0; c < KC; c++) load_block(SB[c], fq, l, BASE + fst * SSTR + KC * fh + c);
    };
    auto fetch_ff2 = [&](int l) {
#pragma unroll
        for (int i = 0; i < TWW; i++) load_block(SA[i], q, l, BASE + fst * SSTR + 4 * KC + (m & 1) * TW + iq0 + i);
    };
    static_assert(TWW <= KC, "the second feed-forward matmul's blocks fit the set");
    auto product = [&](auto swap, const v4i (&w)[8], const uint8_t* from, acc_t acc) -> acc_t {
#pragma unroll
        for (int s = 0; s < 8; s++) acc = frag_mma<decltype(swap)::value>(w[s], *reinterpret_cast<const v4i*>(from + s * FRAG + lane * 16), acc);
        return acc;
    };
    const acc_t zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    // row sums and the quantiser: bf_board.hip.h's, with tiles TWW wave ... owned by a wave in order
    auto xsum = [&](float part, int sl) -> float {
        xch[sl * XS + wave * 64 + lane] = part;
        lds_barrier();
        const float* p = xch + sl * XS + lane;
        return (((p[0] + p[64]) + (p[128] + p[192])) + (p[256] + p[320])) + (p[384] + p[448]);
    };
    auto layernorm = [&](const float (&x)[TWW][16], const float* gamma, const float* beta, float (&y)[TWW][16]) {
        float ts[TWW];
#pragma unroll
        for (int i = 0; i < TWW; i++) {
            float acc = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) acc = acc + x[i][r];
            ts[i] = acc;
        }
        const float s = xsum(TWW == 1 ? ts[0] : ts[0] + ts[TWW - 1], 0);
        const float mean = (s + partner(s, g)) * (1.0f / D);
#pragma unroll
        for (int i = 0; i < TWW; i++) {
            float acc = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float d = x[i][r] - mean;
                acc = __builtin_fmaf(d, d, acc);
            }
            ts[i] = acc;
        }
        const float v = xsum(TWW == 1 ? ts[0] : ts[0] + ts[TWW - 1], 1);
        const float var = (v + partner(v, g)) * (1.0f / D);
        const float rstd = recip_sqrt(var + a.eps);
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f ga = ldg4(gamma + 32 * i + 8 * j + 4 * g);
                const v4f be = ldg4(beta + 32 * i + 8 * j + 4 * g);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float d = x[i][4 * j + k] - mean;
                    y[i][4 * j + k] = __builtin_fmaf(d * rstd, ga[k], be[k]);
                }
            }
    };
    auto quant_exchange = [&](const float (&y)[TWW][16], float (&sa)[KC], bool publish_scales) {
        float am = 0.0f;
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) am = __builtin_fmaxf(am, __builtin_fabsf(y[i][r]));
        xch[2 * XS + wave * 64 + lane] = am;
        lds_barrier();
#pragma unroll
        for (int c = 0; c < KC; c++) {
            float mx = 0.0f;
#pragma unroll
            for (int w = 8 / KC * c; w < 8 / KC * (c + 1); w++) mx = __builtin_fmaxf(mx, xch[2 * XS + w * 64 + lane]);
            mx = __builtin_fmaxf(mx, partner(mx, g));
            sa[c] = mx > 0.0f ? (FP8 ? mx * 0.125f : div127(mx)) : 1.0f;
        }
        if (publish_scales && wave == 0 && g == 0)
#pragma unroll
            for (int c = 0; c < KC; c++) tok[c * 32 + t] = sa[c];
        const Quot by = quot_by(KC == 1 || wave < 4 ? sa[0] : sa[KC - 1]);
#pragma unroll
        for (int i = 0; i < TWW; i++) {
            v4i w;
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = (int)quant4<FP8>(y[i][4 * j], y[i][4 * j + 1], y[i][4 * j + 2], y[i][4 * j + 3], by);
            *reinterpret_cast<v4i*>(act + (TWW * wave + i) * FRAG + lane * 16) = w;
        }
        lds_barrier();
    };
    // wait until `count` flags, `stride` dwords apart, have reached `tag`
    auto wait_flags = [&](int first, int stride, int count, int tag) {
        for (int spins = 0; !dead;) {
            int f = tag;
            if (lane < count) f = (int)__builtin_amdgcn_raw_buffer_load_b32(wsr, lane * (stride * 4), first * 4, SC1);
            if (__all(f - tag >= 0)) break;
            if (++spins > SPIN_LIMIT) dead = true;
            asm volatile("" ::: "memory");
        }
        asm volatile("" ::: "memory");
    };
    // this wave's piece is stored: let the L2 have it, then raise the flag
    auto raise_flag = [&](int at, int tag) {
        wait_vm<0>();
        if (lane == 0 && !dead) __builtin_amdgcn_raw_buffer_store_b32((unsigned)tag, wsr, 0, at * 4, 0);
    };
    auto take = [&](int at) -> v4i { return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wsr, lane16, at, SC1)); };

    // ---- start: parameters and weights of the first layer --------------------------------------------
    if (a.l1 > a.l0) {
        fetch_par(a.l0);
        fetch_qkv(a.l0);
        fetch_out(SB, a.l0, 0);
    }

    // ---- embedding, or the caller's stream -------------------------------------------------------------
    float x[TWW][16];
    const unsigned word = ENC ? (a.taps.alive[(size_t)b * T + t] ? 0u : 0x800u) : a.boards[(size_t)b * T + t];
    const int ctrl = ENC ? 1 : a.control[b];
    const unsigned alive = (unsigned)__ballot(((word >> 11) & 1) == 0 && g == 0);
    if constexpr (ENC) {
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f v = stream_in(a.taps, ((size_t)b * T + t) * D + 32 * (TWW * wave + i) + 8 * j + 4 * g);
#pragma unroll
                for (int k = 0; k < 4; k++) x[i][4 * j + k] = v[k];
            }
    } else {
        const int stm = ctrl < 0;
        int clock = (ctrl < 0 ? -ctrl : ctrl) - 1;
        clock = clock < 0 ? 0 : (clock > 100 ? 100 : clock);
        int rp = a.rep[b];
        rp = rp > 2 ? 2 : rp;
        int ts = ((word >> 6) & 7) * 2 + ((word >> 9) & 1);
        ts = ts > 11 ? 11 : ts;
        const int ct = ((word >> 10) & 1) * 2 + stm;
        const int own = 32 * TWW * wave + 4 * g;
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
                    x[i][4 * j + k] = v + per_board;
                }
            }
    }
    wait_vm<0>();   // the parameters have landed (the next barrier shows them to the other waves)

    for (int l = a.l0; l < a.l1; l++) {
        const int tag = tag0 + (l - a.l0) + 1;
        const int lnext = l + 1 < a.l1 ? l + 1 : l;   // after the last layer its own weights come once more (and are not used)
        const float* const pq = par(l, q);                       // this wave's quarter: parts A and B
        const float* const pB = pq + C::A_FLOATS;

        // ---- LayerNorm 1, quantise ---------------------------------------------------------------------
        float sa[KC];
        {
            float y[TWW][16];
            layernorm(x, pq + C::A_LN1G + 32 * iq0, pq + C::A_LN1B + 32 * iq0, y);
            quant_exchange(y, sa, true);
        }
        if (lnext != l) fetch_par(lnext);   // the other copy's last reads lie before the barriers above

        __builtin_amdgcn_sched_barrier(0);
        // ---- Q, K, V tiles of this member's heads ------------------------------------------------------
        // stored as [lane half g][register r odd][r / 8][token][r / 2 % 4], which is how the 16x16x4 operands are read
        if (tq < 3) {
            const float* const pA = par(l, hq);
            const float sw = pA[C::A_SW + tq * TW + hi];
            acc_t acc[KC];
            float v[16];
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
        if constexpr (TWW == 1) fetch_ff2(l);
        else fetch_out(SA, l, 1);
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
            float p[8];
            float mx = -__builtin_inff();
#pragma unroll
            for (int i = 0; i < 8; i++) {
                float s = sc[i / 4][i % 4] * 0.17677669529663687f;
                s = ((alive >> ch(2 * i + (G >> 1), G & 1)) & 1u) ? s : -__builtin_inff();
                p[i] = s;
                mx = __builtin_fmaxf(mx, s);
            }
            mx = __builtin_fmaxf(mx, partner(mx, g));
            const v2u mr = rows_of(mx);
            mx = __builtin_fmaxf(__int_as_float(mr[0]), __int_as_float(mr[1]));
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
                                                       (G >> 1) * FRAG + ((G & 1) * 32 + c16) * 16, C::WS_A + (tile * 4 + 2 * u) * FRAG + qb * 256, 0);
            raise_flag(C::FLAG_A + tile * 2 + qb, tag);
        }

        // ---- exchange A, output projection + residual --------------------------------------------------
        {
            float o[TWW][16];
            wait_flags(C::FLAG_A + TWW * wave * 2, 1, 2 * TWW, tag);
#pragma unroll
            for (int i = 0; i < TWW; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4f v = __builtin_bit_cast(v4f, take(C::WS_A + ((TWW * wave + i) * 4 + j) * FRAG));
#pragma unroll
                    for (int k = 0; k < 4; k++) o[i][4 * j + k] = v[k];
                }
            float so[KC];
            quant_exchange(o, so, false);
#pragma unroll
            for (int i = 0; i < TWW; i++) {
                acc_t acc[KC];
#pragma unroll
                for (int c = 0; c < KC; c++) acc[c] = product(std::false_type(), i == 0 ? SB[c] : SA[c], act + 8 * c * FRAG, zero);
                if (i == 0) fetch_ff1(l);
                v4f bo[4];
                load_tile16(pq + C::A_BOUT + 32 * (iq0 + i), g, bo);
                const float sw = pq[C::A_SW + 3 * TW + iq0 + i];
#pragma unroll
                for (int r = 0; r < 16; r++) x[i][r] = x[i][r] + (chunk_sum<KC, false>(acc, r, so) * sw + bo[r / 4][r % 4]);
                pin16(x[i]);
            }
            if constexpr (TWW > 1) fetch_ff2(l);
        }

        __builtin_amdgcn_sched_barrier(0);
        // ---- LayerNorm 2, quantise, this member's chunk of the hidden row ---------------------------------
        {
            float y[TWW][16];
            layernorm(x, pB + C::B_LN2G + 32 * iq0, pB + C::B_LN2B + 32 * iq0, y);
            quant_exchange(y, sa, false);
        }
        __builtin_amdgcn_sched_barrier(0);
        float sh;
        {
            const float* const pF = par(l, fq) + C::A_FLOATS;
            acc_t acc[KC];
#pragma unroll
            for (int c = 0; c < KC; c++) acc[c] = product(std::false_type(), SB[c], act + 8 * c * FRAG, zero);
            v4f b1[4];
            load_tile16(pF + C::B_BFF1 + 128 * fst + 32 * fh, g, b1);
            const float sw1 = pF[C::B_SW + 4 * fst + fh];
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
            mx = __builtin_fmaxf(mx, partner(mx, g));
            sh = mx > 0.0f ? (FP8 ? mx * 0.125f : div255(mx)) : 1.0f;
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
            acc_t own[TWW];
            const int mine = C::WS_B + (m * 8 + wave) * C::B_PIECE;
#pragma unroll
            for (int i = 0; i < TWW; i++) {
                acc_t init = zero;
                if constexpr (!FP8) {   // 128 * sum(w): the offset of the unsigned bytes stored as q - 128
                    v4i w0[4];
                    load_tile16i(pB + C::B_WSUM + m * CW + 32 * (iq0 + i), g, w0);
#pragma unroll
                    for (int r = 0; r < 16; r++) init[r] = w0[r / 4][r % 4];
                }
                own[i] = product(std::false_type(), SA[i], hid, init);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    __builtin_amdgcn_raw_buffer_store_b128(v4i{accbits(own[i], 4 * j), accbits(own[i], 4 * j + 1), accbits(own[i], 4 * j + 2), accbits(own[i], 4 * j + 3)},
                                                           wsr, lane16, mine + (4 * i + j) * FRAG, 0);
            }
            __builtin_amdgcn_raw_buffer_store_b32((unsigned)__float_as_int(sh), wsr, lane * 4, mine + 4 * TWW * FRAG, 0);
            raise_flag(C::FLAG_B + m * 8 + wave, tag);
            wait_flags(C::FLAG_B + wave, 8, NWG, tag);
            float shc[NWG];
#pragma unroll
            for (int c = 0; c < NWG; c++)
                shc[c] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(wsr, lane * 4, C::WS_B + (c * 8 + wave) * C::B_PIECE + 4 * TWW * FRAG, SC1));
#pragma unroll
            for (int i = 0; i < TWW; i++) {
                double o64[16];
                float o32[16];
#pragma unroll
                for (int c0 = 0; c0 < NWG; c0 += 4) {   // four members' pieces in flight
                    __builtin_amdgcn_sched_barrier(0);
                    v4i piece[4][4];
#pragma unroll
                    for (int u = 0; u < 4; u++)
#pragma unroll
                        for (int j = 0; j < 4; j++) piece[u][j] = take(C::WS_B + ((c0 + u) * 8 + wave) * C::B_PIECE + (4 * i + j) * FRAG);
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int c = c0 + u;
                        if constexpr (FP8) {
                            const float sw = pB[C::B_SW + 16 + (iq0 + i) * KCF + c];
#pragma unroll
                            for (int r = 0; r < 16; r++) {
                                const float part = (__int_as_float(piece[u][r / 4][r % 4]) * shc[c]) * sw;
                                o32[r] = c == 0 ? part : o32[r] + part;
                            }
                        } else {
                            const double sc = (double)shc[c];
#pragma unroll
                            for (int r = 0; r < 16; r++) {
                                const double full = (double)piece[u][r / 4][r % 4];
                                o64[r] = c == 0 ? full * sc : __builtin_fma(full, sc, o64[r]);
                            }
                        }
                    }
                }
                v4f b2[4];
                load_tile16(pB + C::B_BFF2 + 32 * (iq0 + i), g, b2);
                const float sw = pB[C::B_SW + 16 + iq0 + i];
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float upd;
                    if constexpr (FP8) upd = o32[r] + b2[r / 4][r % 4];
                    else upd = (float)o64[r] * sw + b2[r / 4][r % 4];
                    x[i][r] = x[i][r] + upd;
                }
                if (dead)
#pragma unroll
                    for (int r = 0; r < 16; r++) x[i][r] = __builtin_nanf("");
                pin16(x[i]);
            }
            fetch_qkv(lnext);
            fetch_out(SB, lnext, 0);
        }
    }
    if (wave == 0 && lane == 0) flags[m] = tag0 + (a.l1 - a.l0);

    if constexpr (ENC) {
        if (m == 0)
#pragma unroll
            for (int i = 0; i < TWW; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    stream_out(a.taps, ((size_t)b * T + t) * D + 32 * (TWW * wave + i) + 8 * j + 4 * g,
                               v4f{x[i][4 * j], x[i][4 * j + 1], x[i][4 * j + 2], x[i][4 * j + 3]});
        return;
    }

    // ---- final norm and heads: member 0 the policy, member 1 promotion and value -------------------------
    if (m > 1) return;
    const int G = lane >> 4, c16 = lane & 15;
    // the head tile's fragments, HEAD_SET of them; the first ones now
    constexpr int HEAD_SET = 32;
    static_assert(8 * HB % HEAD_SET == 0, "whole sets");
    v4i hw[HEAD_SET];
    auto load_head = [&](int ht, int rh, int f0) {
        const int at = (ht * stride_q + a.n_layers * BPW) * BLOCK + f0 * FRAG, lane_at = (16 * rh + c16 + 32 * (G & 1)) * 16;
#pragma unroll
        for (int f = 0; f < HEAD_SET; f++)
            hw[f] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane_at + f % 4 * FRAG, at + f / 4 * 4 * FRAG, 0));
    };
    if (m == 0) load_head(wave >> 2, (wave >> 1) & 1, 0);
    else if (wave < 2) load_head(2, 0, 0);
    float hn[TWW][16];
    layernorm(x, gp + C::G_NFG + 32 * TWW * wave, gp + C::G_NFB + 32 * TWW * wave, hn);
    float* const hnb = qkv;
    auto publish = [&](const float (&v)[TWW][16]) {
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                *reinterpret_cast<v4f*>(hnb + (((TWW * wave + i) * 4 + j) * 64 + lane) * 4) = v4f{v[i][4 * j], v[i][4 * j + 2], v[i][4 * j + 1], v[i][4 * j + 3]};
    };
    publish(hn);
    lds_barrier();
    // (elements 0 and 2 of a register quad lie together, as do 1 and 3.)
    // Rows 16 rh .. of head tile `ht` times tokens 16 th ..: the chain of the 32x32x2 form, two of whose steps (four k) are
    // one step here.  Lane (row or token, k) takes element k / 2 and 2 + k / 2 of the fragment lane of half k % 2.
    auto head_product = [&](int ht, int rh, int th) -> v4f {
        const float* hp = hnb + (16 * th + c16 + 32 * (G & 1)) * 4 + 2 * (G >> 1);
        const bool up = G >> 1;
        v4f acc = {0, 0, 0, 0};
#pragma unroll
        for (int f0 = 0; f0 < 8 * HB; f0 += HEAD_SET) {
            if (f0) load_head(ht, rh, f0);
#pragma unroll
            for (int f = 0; f < HEAD_SET; f++) {
                const v4f w = __builtin_bit_cast(v4f, hw[f]);
                const v2f h = *reinterpret_cast<const v2f*>(hp + (f0 + f) * 256);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(up ? w[1] : w[0], h[0], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(up ? w[3] : w[2], h[1], acc, 0, 0, 0);
            }
        }
        return acc;
    };
    if (m == 0) {
        // policy: squares 32 ht + 16 rh + 4 G .. of token 16 th + c16, optional legal-move AND and argmax
        const int ht = wave >> 2, rh = (wave >> 1) & 1, th = wave & 1, tk = 16 * th + c16, sq0 = 32 * ht + 16 * rh + 4 * G;
        unsigned long long mw = ~0ull;
        if (a.mask) mw = a.mask[(size_t)b * T + tk];
        const v4f hd = head_product(ht, rh, th);
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
            auto better = [](float ov, int oi, float bv_, int bi_) {   // larger, lowest index on ties; no move at all is worst
                return oi != 0x7fffffff && (bi_ == 0x7fffffff || ov > bv_ || (ov == bv_ && oi < bi_));
            };
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                const float ov = __shfl_xor(bv, d);
                const int oi = __shfl_xor(bi, d);
                const bool tk_ = better(ov, oi, bv, bi);
                bv = tk_ ? ov : bv;
                bi = tk_ ? oi : bi;
            }
            if (lane == 0) {
                xch[2 * XS + wave * 2] = bv;
                xch[2 * XS + wave * 2 + 1] = __int_as_float(bi);
            }
            lds_barrier();
            if (wave == 0 && lane == 0) {
#pragma unroll
                for (int w = 1; w < 8; w++) {
                    const float ov = xch[2 * XS + w * 2];
                    const int oi = __float_as_int(xch[2 * XS + w * 2 + 1]);
                    const bool tk_ = better(ov, oi, bv, bi);
                    bv = tk_ ? ov : bv;
                    bi = tk_ ? oi : bi;
                }
                a.best[b] = bi == 0x7fffffff ? -1 : bi;
            }
        }
        return;
    }
    auto value_of = [&](const v4f& hd) -> float {
        if (a.n_value == 1) return tanh_dev(hd[0]);
        const float r0 = hd[0], r1 = hd[1], r2 = hd[2];   // classes loss, draw, win
        const float mx = __builtin_fmaxf(__builtin_fmaxf(r0, r1), r2);
        const float e0 = exp_neg(r0 - mx), e1 = exp_neg(r1 - mx), e2 = exp_neg(r2 - mx);
        return (e2 - e0) / ((e0 + e1) + e2);
    };
    // rows 0..3 of head tile 2 are the promotion rows (lane row 0), rows 4.. the value rows (lane row 1)
    if (wave < 2) {
        const v4f hd = head_product(2, 0, wave);
        const int tk = 16 * wave + c16;
        if (G == 0) {
            const size_t at = ((size_t)b * T + tk) * 4;
            if (a.out_fp32) *reinterpret_cast<v4f*>((float*)a.promo + at) = hd;
            else *reinterpret_cast<v4h*>((_Float16*)a.promo + at) = v4h{(_Float16)hd[0], (_Float16)hd[1], (_Float16)hd[2], (_Float16)hd[3]};
        }
        if (a.vmode == 0 && G == 1 && tk == (ctrl < 0 ? 31 : 15)) a.value[b] = value_of(hd);
    }
    // pooled heads: the mean over the live tokens of the normalised stream (1), or the final norm of the mean of the
    // residual stream (2), through the value rows like a token; White's frame, so negated when Black is to move
    if (a.vmode != 0) {
        float pv[TWW][16];
        const bool lv = (alive >> t) & 1u;
        const float cdiv = (float)(__builtin_popcount(alive) > 0 ? __builtin_popcount(alive) : 1);
#pragma unroll
        for (int i = 0; i < TWW; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                float v = lv ? (a.vmode == 1 ? hn[i][r] : x[i][r]) : 0.0f;
#pragma unroll
                for (int d = 16; d >= 1; d >>= 1) v = v + __shfl_xor(v, d);
                pv[i][r] = v / cdiv;
            }
        if (a.vmode == 2) {
            float hv[TWW][16];
            layernorm(pv, gp + C::G_NFG + 32 * TWW * wave, gp + C::G_NFB + 32 * TWW * wave, hv);
#pragma unroll
            for (int i = 0; i < TWW; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) pv[i][r] = hv[i][r];
        }
        lds_barrier();   // every wave has finished reading the normalised stream
        publish(pv);
        lds_barrier();
        if (wave == 0) {
            if constexpr (8 * HB > HEAD_SET) load_head(2, 0, 0);   // else they are still there
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
