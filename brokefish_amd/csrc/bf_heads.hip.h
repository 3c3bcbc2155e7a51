// The heads of the evaluators that hold one or two positions in a workgroup of eight wavefronts (bf_duo.hip.h, bf_wide.hip.h): their
// products, the stores, the best move and the pooled value.
//
// The products come in pieces of 16 rows of a head tile and 16 tokens (v_mfma_f32_16x16x4f32: the fused-multiply-add chain of
// the 32x32x2 form, four links a step).  A wave takes 16 rows of a policy tile for both halves of its position's tokens
// (one position: for one half), and one wave of each SIMD (one position: of two) a half of a position's tokens with the first rows of
// tile 2, where promotion and value lie.  256 wide, two positions, that is 10.2 k clocks of every SIMD; as 32x32 products of
// whole tiles (tile 2's 25 rows of zeros among them) it was 16.4 k of three SIMDs, and the fourth idled.  With the final norm's
// parameters and the legal moves asked for ahead and the best move found without LDS permutations: phases heads + stores 29.9 k ->
// 23.5 k ticks of 462 k; 300 positions 171.2 -> 168.2 us, 100 114.9 -> 113.8, 4096 1427 -> 1411, e4m3 300 230.6 -> 228.4, 4096 1901 -> 1891.
#pragma once

#include "bf_board.hip.h"

typedef float v2f __attribute__((ext_vector_type(2)));

namespace bf {

// NP positions; head tiles of 8 HB fragments, RING of them in flight
template <int NP, int HB, int RING>
struct Heads {
    static constexpr int FRAGS = 8 * HB, HALVES = NP, NONE = 0x7fffffff;   // HALVES: token halves of a policy wave
    static constexpr int EARLY = 4;                                        // operands come from LDS this many fragments early
    static constexpr int SET = 8;                                          // fragments of a set in the pooled heads
    static_assert(RING <= FRAGS && SET <= RING && FRAGS % SET == 0, "the first loads stay inside the tile; whole sets");

    const KArgs& a;
    const int lane, q, sub, G, c16;
    const int ht, rh, th0;                      // the policy rows 16 rh .. of head tile ht; its first token half
    const int mine;                             // of the workgroup's positions
    const bool extra;                           // has a piece of tile 2: of position xmine, token half xth
    const int xmine, xth;
    const int b, xb, xctrl;
    const bool live, xlive;
    const int stream_at, stream_p;              // the published stream in LDS, and a position's share of it, bytes
    const int from0, from;
    __amdgpu_buffer_rsrc_t policy_tile, tile2;
    v4i w[RING];
    unsigned long long legal[HALVES];
    v4f head[HALVES], rest;

    // by value: chosen as an element of the array, it was put into private memory (512 wide: 12 bytes a lane, 33 MiB written by 16384 positions)
    static __device__ __forceinline__ int of(int p, int first, int second) { return p ? second : first; }
    __device__ __forceinline__ Heads(const KArgs& a_, int blocks_per_layer, int lane_, int wave, const int (&bp)[NP], const bool (&live_)[NP], const int (&ctrl)[NP],
                                     int stream_at_, int stream_p_)
        : a(a_), lane(lane_), q(wave & 3), sub(wave >> 2), G(lane_ >> 4), c16(lane_ & 15), ht(q & 1), rh(q >> 1), th0(NP == 2 ? 0 : sub), mine(NP == 2 ? sub : 0),
          extra(sub == 1 && (NP == 2 || q < 2)), xmine(NP == 2 ? q & 1 : 0), xth(NP == 2 ? q >> 1 : q), b(mine ? bp[NP - 1] : bp[0]), xb(xmine ? bp[NP - 1] : bp[0]),
          xctrl(of(xmine, ctrl[0], ctrl[NP - 1])), live(mine ? live_[NP - 1] : live_[0]), xlive(xmine ? live_[NP - 1] : live_[0]), stream_at(stream_at_),
          // Lane (row, k) reads, of a fragment, the lane of its row and of half k % 2, from element k / 2 on: what it multiplies lies in places
          // 0 and 2 then.  (The last lanes' reads end four bytes behind the fragment, in the next one or the block of padding.)
          stream_p(stream_p_), from0((c16 + 32 * (G & 1)) * 16 + 4 * (G >> 1)), from(from0 + 256 * rh) {
        // A wave without a piece of tile 2 sees it empty, and its loads move nothing: with a branch around them the number of loads under way
        // would not be known, and the chains behind would wait for all of them at every step (577 positions 283.5 -> 282.7 us; 100 and 200
        // as before).
        const size_t stride = (size_t)a.n_layers * blocks_per_layer + HB + 1;
        auto tile = [&](int n, bool used) {
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.wstream + (n * stride + (size_t)a.n_layers * blocks_per_layer) * BLOCK), 0,
                                                     used ? HB * BLOCK + 16 : 0, 0x00027000);
        };
        policy_tile = tile(ht, true);
        tile2 = tile(2, extra);
    }

    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& tile, int lane_at, int f, int at) {
        w[at] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(tile, lane_at, f * FRAG, 0));
    }
    // the first fragments and the legal moves, ahead of their use
    __device__ __forceinline__ void ask() {
#pragma unroll
        for (int j = 0; j < RING; j++) load(policy_tile, from, j, j);
#pragma unroll
        for (int i = 0; i < HALVES; i++) legal[i] = a.mask ? a.mask[(size_t)b * T + 16 * (th0 + i) + c16] : ~0ull;
    }
    // tile `tile` of position p's normalised stream as operand fragments: lane (t, g) holds the four floats of register quad j,
    // elements 0 and 2 together
    __device__ __forceinline__ void publish(int p, int tile, const float (&v)[16]) const {
        uint8_t* const to = board::lds + stream_at + p * stream_p + tile * 4 * FRAG + lane * 16;
#pragma unroll
        for (int j = 0; j < 4; j++) *reinterpret_cast<v4f*>(to + j * FRAG) = v4f{v[4 * j], v[4 * j + 2], v[4 * j + 1], v[4 * j + 3]};
    }
    // lane (token, k) of a step: element k / 2 (and 2 + k / 2 in the next step) of the fragment lane of half k % 2
    __device__ __forceinline__ const uint8_t* operands(int p, int th) const {
        int at = stream_at + p * stream_p + (32 * (G & 1) + 16 * th + c16) * 16 + 8 * (G >> 1);
        asm volatile("" : "+v"(at));   // one address register; the rest are the instructions' own offsets
        return board::lds + at;
    }
    static __device__ __forceinline__ v2f operand(const uint8_t* of, int half, int f) { return *reinterpret_cast<const v2f*>(of + f * FRAG + half * 256); }
    static __device__ __forceinline__ void steps(const v4i& wi, const v2f& h, v4f& acc) {
        const v4f wf = __builtin_bit_cast(v4f, wi);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[0], h[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[2], h[1], acc, 0, 0, 0);
    }
    __device__ __forceinline__ void products() {
#pragma unroll
        for (int i = 0; i < HALVES; i++) head[i] = v4f{0, 0, 0, 0};
        rest = v4f{0, 0, 0, 0};
        {
            const uint8_t* const of = operands(mine, th0);
            v2f h[EARLY][HALVES];
#pragma unroll
            for (int f = 0; f < EARLY; f++)
#pragma unroll
                for (int i = 0; i < HALVES; i++) h[f][i] = operand(of, i, f);
#pragma unroll
            for (int f = 0; f < FRAGS; f++) {
#pragma unroll
                for (int i = 0; i < HALVES; i++) {
                    steps(w[f % RING], h[f % EARLY][i], head[i]);
                    if (f + EARLY < FRAGS) h[f % EARLY][i] = operand(of, i, f + EARLY);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (f + RING < FRAGS) load(policy_tile, from, f + RING, f % RING);
                else load(tile2, from0, f + RING - FRAGS, (f + RING) % RING);
            }
        }
        if (extra) {
            const uint8_t* const of = operands(xmine, xth);
            v2f h[EARLY];
#pragma unroll
            for (int f = 0; f < EARLY; f++) h[f] = operand(of, 0, f);
#pragma unroll
            for (int f = 0; f < FRAGS; f++) {
                steps(w[(FRAGS + f) % RING], h[f % EARLY], rest);
                if (f + EARLY < FRAGS) h[f % EARLY] = operand(of, 0, f + EARLY);
                __builtin_amdgcn_sched_barrier(0);
                if (f + RING < FRAGS) load(tile2, from0, f + RING, (FRAGS + f) % RING);
            }
        }
    }
    __device__ __forceinline__ float value_of(const v4f& hd) const {
        if (a.n_value == 1) return tanh_dev(hd[0]);
        const float r0 = hd[0], r1 = hd[1], r2 = hd[2];   // classes loss, draw, win
        const float mx = __builtin_fmaxf(__builtin_fmaxf(r0, r1), r2);
        const float e0 = exp_neg(r0 - mx), e1 = exp_neg(r1 - mx), e2 = exp_neg(r2 - mx);
        return (e2 - e0) / ((e0 + e1) + e2);
    }
    // `met`: 64 bytes of LDS for the waves' best moves, which nobody reads or writes any more
    template <typename BARRIER>
    __device__ __forceinline__ void store(void* met_, BARRIER&& barrier) {
        // tile 2: rows 64 .. 67 (lanes G = 0) are the promotions, rows 68 .. 70 (G = 1) the value, whose token is the mover's king
        if (extra && xlive) {
            const int tk = 16 * xth + c16;
            if (a.vmode == 0 && G == 1 && tk == (xctrl < 0 ? 31 : 15)) a.value[xb] = value_of(rest);
            if (G == 0) {
                const size_t at = ((size_t)xb * T + tk) * 4;
                if (a.out_fp32) *reinterpret_cast<v4f*>((float*)a.promo + at) = rest;
                else *reinterpret_cast<v4h*>((_Float16*)a.promo + at) = v4h{(_Float16)rest[0], (_Float16)rest[1], (_Float16)rest[2], (_Float16)rest[3]};
            }
        }
        // policy: squares 32 ht + 16 rh + 4 G .. of the wave's tokens, optional legal-move AND and argmax
        float bv = -__builtin_inff();
        int bi = NONE;
        const int sq0 = 32 * ht + 16 * rh + 4 * G;
#pragma unroll
        for (int i = 0; i < HALVES; i++) {
            const int tk = 16 * (th0 + i) + c16;
            const unsigned ok = (unsigned)(legal[i] >> sq0);
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const bool is = (ok >> k) & 1u;
                v[k] = is ? head[i][k] : -__builtin_inff();
                // a lane visits its moves in increasing order, so '>' keeps the lowest
                if (is && (bi == NONE || v[k] > bv)) { bv = v[k]; bi = tk * 64 + sq0 + k; }
            }
            const size_t at = ((size_t)b * T + tk) * 64 + sq0;
            if (live) {
                if (a.out_fp32) *reinterpret_cast<v4f*>((float*)a.policy + at) = v4f{v[0], v[1], v[2], v[3]};
                else *reinterpret_cast<v4h*>((_Float16*)a.policy + at) = v4h{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
            }
        }
        if (!a.mask || !a.best) return;
        auto merge = [&](float ov, int oi) {
            const bool take = oi != NONE && (bi == NONE || ov > bv || (ov == bv && oi < bi));
            bv = take ? ov : bv;
            bi = take ? oi : bi;
        };
        auto over_dpp = [&](auto ctrl) {   // another lane of the row of 16
            constexpr int c = decltype(ctrl)::value;
            const int ov = __builtin_amdgcn_update_dpp(0, __float_as_int(bv), c, 0xf, 0xf, true), oi = __builtin_amdgcn_update_dpp(0, bi, c, 0xf, 0xf, true);
            merge(__int_as_float(ov), oi);
        };
        auto over_swap = [&](auto swap) {   // both lanes get both values and keep the better one
            const auto v2 = swap(__float_as_int(bv)), i2 = swap(bi);
            bv = __int_as_float((int)v2[0]);
            bi = (int)i2[0];
            merge(__int_as_float((int)v2[1]), (int)i2[1]);
        };
        over_dpp(std::integral_constant<int, 0xb1>());    // xor 1
        over_dpp(std::integral_constant<int, 0x4e>());    // xor 2
        over_dpp(std::integral_constant<int, 0x141>());   // the mirrored eight
        over_dpp(std::integral_constant<int, 0x140>());   // the mirrored sixteen
        over_swap([](int v) { return __builtin_amdgcn_permlane16_swap(v, v, false, false); });
        over_swap([](int v) { return __builtin_amdgcn_permlane32_swap(v, v, false, false); });
        int* const met = static_cast<int*>(met_);
        if (lane == 0) {
            met[2 * (4 * sub + q)] = __float_as_int(bv);
            met[2 * (4 * sub + q) + 1] = bi;
        }
        barrier();
        if (q == 0 && (NP == 2 || sub == 0) && live) {
#pragma unroll
            for (int o = 1; o < 8 / NP; o++) merge(__int_as_float(met[2 * (4 * mine + o)]), met[2 * (4 * mine + o) + 1]);
            if (lane == 0) a.best[b] = bi == NONE ? -1 : bi;
        }
    }
    // tile 2's rows once more, against the pooled rows, published meanwhile (every token column holds the same row), in the same order
    __device__ __forceinline__ void pooled() {
        if (!extra || xth != 0) return;
        v4f hd = {0, 0, 0, 0};
        const uint8_t* const of = operands(xmine, 0);
        for (int f0 = 0; f0 < FRAGS; f0 += SET) {
#pragma unroll
            for (int j = 0; j < SET; j++) load(tile2, from0, f0 + j, j);
#pragma unroll
            for (int j = 0; j < SET; j++) steps(w[j], operand(of, 0, f0 + j), hd);
        }
        if (lane == 16 && xlive) {
            const float v = value_of(hd);
            a.value[xb] = xctrl > 0 ? v : -v;
        }
    }
};

}  // namespace bf
