// Edge expansion behind the evaluator: logits + legal-move words -> the edges of a search node.
//
// For every position: enumerate the set bits of the 32 legal-move words in canonical order
// (ascending slot, then square; a pawn move onto the last rank fans out into four edges in the
// order N B R Q), give each edge the unnormalised log-prior
//     policy[slot][square]  (+ log_softmax(promo[slot])[type] for a promotion edge),
// keep the E largest if there are more than E (ties by canonical order, survivors stay in
// canonical order), softmax over the survivors, and write move codes, fp16 priors, the edge
// count, the mass dropped by the truncation and the value mapped from [-1,1] to [0,1].
// Restates reference docs/reference/search.md:616-636 and brokefish/search/torch_impl.py:962-1033.
//
// Two positions per wavefront, 32 lanes each: lane s of a half owns the mask word of slot s, so lane order
// is canonical order and a slot's first edge index is a prefix sum over the half.  Candidates (some 31
// per position) are then taken one per lane, 32 a round: a lane finds the slot its candidate belongs to
// by a running maximum over the slots' first indices and the square as the k-th set bit of that
// slot's word -- no loop over bits -- and fetches its one logit straight from the policy row (the loop,
// with the logits it might need staged in LDS, remains for wavefronts in which a pawn promotes).
// Reductions run over DPP and lane swaps, ranks and counts over ballots; the edges are put together in
// LDS and leave as whole 16-byte pieces.  The truncation threshold (the E-th largest log-prior) is
// found by bisection on the ordered bit pattern of the float.  More than 128 candidates of a position take a
// second build of the same code with twice the rounds (5000 positions of 218 moves: 15 us; holding all of them to
// its size would cost the others 8 %, 20 % where rows truncate), more than 256 (no legal position, an
// arbitrary mask) the whole wavefront for the one position, every pass walking the bits again (184 us).
// Bound by instruction issue and, from some 16384 positions on, by HBM; one position per wavefront with
// staged logits took 48 us for 65536 positions (E = 96), this 23 us (4 TB/s of its bytes).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <cstdint>
#include <cstdio>

#include "bf_args.h"
#include "bf_movegen.hip.h"

namespace {

constexpr int PAWN = 0;          // reference docs/reference/spec.md:47
constexpr int PROMO_SHIFT = 11;  // brokefish/search/torch_impl.py:61-62

struct KExpand {
    const void* policy;
    const void* promo;
    const float* value;
    const uint64_t* mask;
    const uint16_t* boards;
    const int16_t* control;
    const uint8_t* active;
    const int* leaf_index;        // optional compacted list: slot j expands position leaf_index[j] for j < *leaf_count
    const int* leaf_count;
    int n, E, logits_fp32;
    int whole_rows;               // a row of edges is whole 16-byte pieces, and few enough to be put together in LDS
    int16_t* edge_move;
    _Float16* edge_prior;
    int* n_edges;
    int* count;
    float* dropped;
    _Float16* node_value;
    uint64_t* mask_out;           // legal-move words and check flags that are generated here (`mask` is then mask_out)
    uint8_t* in_check;
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
    return v;
}
__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
    return v;
}
// exclusive prefix sum over the 64 lanes
__device__ __forceinline__ int wave_exclusive(int v, int lane) {
    int inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(inc, d);
        if (lane >= d) inc += o;
    }
    return inc - v;
}
// bit pattern whose unsigned order is the order of the floats (-0 + 0 is 0: the two zeros are one value)
__device__ __forceinline__ unsigned ordered(float f) {
    const unsigned u = __float_as_uint(f + 0.0f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
// what one lane of this wave wrote to LDS is read by another: LDS operations of a wave are carried
// out in program order, the fences keep the compiler from changing that order
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- operations within a half (32 lanes) of the wavefront ---------------------------------------------
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp0(int v) {   // 0 where no lane supplies a value
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, true);
}
constexpr int ROW_SHR = 0x110, ROW_ROR = 0x120, ROW_BCAST15 = 0x142;
// inclusive scans: within a row of sixteen, then the first row's last lane into the second row
__device__ __forceinline__ int half_scan_add(int v) {
    v += dpp0<ROW_SHR + 1>(v);
    v += dpp0<ROW_SHR + 2>(v);
    v += dpp0<ROW_SHR + 4>(v);
    v += dpp0<ROW_SHR + 8>(v);
    v += dpp0<ROW_BCAST15, 0xa>(v);
    return v;
}
__device__ __forceinline__ int half_scan_max(int v) {   // of values >= 0
    v = max(v, dpp0<ROW_SHR + 1>(v));
    v = max(v, dpp0<ROW_SHR + 2>(v));
    v = max(v, dpp0<ROW_SHR + 4>(v));
    v = max(v, dpp0<ROW_SHR + 8>(v));
    v = max(v, dpp0<ROW_BCAST15, 0xa>(v));
    return v;
}
template <typename OP>
__device__ __forceinline__ float half_reduce(float v, OP op) {   // the result in every lane of the half
    v = op(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), ROW_ROR + 8, 0xf, 0xf, false)));
    v = op(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), ROW_ROR + 4, 0xf, 0xf, false)));
    v = op(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), ROW_ROR + 2, 0xf, 0xf, false)));
    v = op(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), ROW_ROR + 1, 0xf, 0xf, false)));
    const int i = __float_as_int(v);
    const auto r = __builtin_amdgcn_permlane16_swap(i, i, false, false);
    return op(__int_as_float(r[0]), __int_as_float(r[1]));
}
__device__ __forceinline__ float half_max(float v) { return half_reduce(v, [](float x, float y) { return fmaxf(x, y); }); }
__device__ __forceinline__ float half_sum(float v) { return half_reduce(v, [](float x, float y) { return x + y; }); }
// lanes of this half below this one whose bit is set in a ballot
__device__ __forceinline__ int half_below(unsigned long long ballot, int half) {
    return half ? __builtin_amdgcn_mbcnt_hi((unsigned)(ballot >> 32), 0) : __builtin_amdgcn_mbcnt_lo((unsigned)ballot, 0);
}
// position of the k-th (from 0) set bit of a 64-bit word
__device__ __forceinline__ int kth_bit(unsigned lo, unsigned hi, int k) {
    int c = __popc(lo);
    const bool up = k >= c;
    unsigned x = up ? hi : lo;
    int at = up ? 32 : 0;
    k -= up ? c : 0;
#pragma unroll
    for (int w = 16; w >= 1; w >>= 1) {
        c = __popc(x & ((1u << w) - 1u));
        const bool t = k >= c;
        k -= t ? c : 0;
        x = t ? x >> w : x;
        at += t ? w : 0;
    }
    return at;
}

constexpr int EXPAND_WAVES = 4;       // wavefronts per workgroup
// Candidates of a position in the two-position form, 32 per round: a wavefront in which a position has more than the few
// rounds hold (128; random games have 31, a board of queens up to 218) runs the form of eight rounds.
constexpr int FEW_ROUNDS = 4, MOST_ROUNDS = 8;
constexpr int CAND_CAP = 32 * MOST_ROUNDS;

struct Shared {   // a half's part of the LDS
    int16_t* code;
    _Float16* prior;
    float* add;          // promotion log-probability of a candidate
    unsigned* owner;     // one byte per candidate
};

template <bool FP32>
__device__ __forceinline__ float logit(const void* p, size_t i) {
    return FP32 ? ((const float*)p)[i] : (float)((const _Float16*)p)[i];
}
// log_softmax of a slot's four promotion logits
template <bool FP32>
__device__ __forceinline__ void promotion_logs(const void* promo, size_t slot, float (&lp)[4]) {
    float x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = logit<FP32>(promo, slot * 4 + k);
    const float mx = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
    const float s = ((__expf(x[0] - mx) + __expf(x[1] - mx)) + __expf(x[2] - mx)) + __expf(x[3] - mx);
    const float ls = __logf(s);
#pragma unroll
    for (int k = 0; k < 4; k++) lp[k] = (x[k] - mx) - ls;
}
__device__ __forceinline__ void write_counts(const KExpand& a, int b, int n_edges, int total, bool trunc, float s_all, float s_keep) {
    a.n_edges[b] = n_edges;
    if (a.count) a.count[b] = total;
    if (a.dropped) a.dropped[b] = trunc ? (s_all - s_keep) / s_all : 0.0f;
    if (a.node_value) a.node_value[b] = (_Float16)((a.value[b] + 1.0f) / 2.0f);
}

// One position on the whole wavefront, any number of candidates: lane l owns half a mask word (slot l / 2,
// squares 32 * (l % 2) .. + 31), nothing is stored per candidate, every pass walks the lane's bits again.
template <bool FP32>
__device__ void expand_many(const KExpand& a, int b, int lane) {
    const int p = lane >> 1, half = lane & 1;
    const unsigned word = a.boards[(size_t)b * 32 + p];
    const int ctrl = a.control[b];
    const bool pawn = ((word >> 11) & 1u) == 0 && ((word >> 6) & 7u) == PAWN;
    const uint64_t m64 = a.mask[(size_t)b * 32 + p];
    const unsigned mh = half ? (unsigned)(m64 >> 32) : (unsigned)m64;
    const unsigned last = ctrl < 0 ? (half == 0 ? 0xFFu : 0u) : (half == 1 ? 0xFF000000u : 0u);
    const unsigned pr = pawn ? (mh & last) : 0u;
    const int total = wave_sum((int)(__popc(mh) + 3 * __popc(pr)));
    float lp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (pr) promotion_logs<FP32>(a.promo, (size_t)b * 32 + p, lp);
    // visit this lane's candidates in canonical order: f(log-prior, move code)
    auto each = [&](auto&& f) {
        unsigned m = mh;
        while (m) {
            const int i = __builtin_ctz(m);
            m &= m - 1;
            const int mv = p * 64 + 32 * half + i;
            const float l = logit<FP32>(a.policy, (size_t)b * 2048 + mv);
            if ((pr >> i) & 1u) {
#pragma unroll
                for (int k = 0; k < 4; k++) f(l + lp[k], mv | (k << PROMO_SHIFT));
            } else {
                f(l, mv);
            }
        }
    };
    int16_t* const em = a.edge_move + (size_t)b * a.E;
    _Float16* const ep = a.edge_prior + (size_t)b * a.E;
    const bool trunc = total > a.E;
    float mx = -INFINITY;
    each([&](float l, int) { mx = fmaxf(mx, l); });
    mx = wave_max(mx);
    unsigned T = 0;   // ordered pattern of the E-th largest log-prior, `need` ties at T survive
    int need = 0, tie_before = 0;
    if (trunc) {
#pragma clang loop unroll(disable)
        for (int bit = 31; bit >= 0; bit--) {
            const unsigned cand = T | (1u << bit);
            int c = 0;
            each([&](float l, int) { c += ordered(l) >= cand; });
            if (wave_sum(c) >= a.E) T = cand;
        }
        int gt = 0, eq = 0;
        each([&](float l, int) {
            const unsigned o = ordered(l);
            gt += o > T;
            eq += o == T;
        });
        need = a.E - wave_sum(gt);
        tie_before = wave_exclusive(eq, lane);
    }
    // one pass: kept count of this lane, softmax denominators over all and over the survivors
    int kept = 0, tie = tie_before;
    float sa = 0.0f, sk = 0.0f;
    each([&](float l, int) {
        const float e = __expf(l - mx);
        sa += e;
        bool keep = true;
        if (trunc) {
            const unsigned o = ordered(l);
            keep = o > T || (o == T && tie < need);
            tie += o == T;
        }
        if (keep) { kept++; sk += e; }
    });
    const float s_all = wave_sum(sa), s_keep = wave_sum(sk);
    int pos = wave_exclusive(kept, lane);
    const int n_edges = __shfl(pos + kept, 63);
    // write the survivors in canonical order
    const float inv = 1.0f / s_keep;
    tie = tie_before;
    each([&](float l, int code) {
        bool keep = true;
        if (trunc) {
            const unsigned o = ordered(l);
            keep = o > T || (o == T && tie < need);
            tie += o == T;
        }
        if (keep) {
            em[pos] = (int16_t)code;
            ep[pos] = (_Float16)(__expf(l - mx) * inv);
            pos++;
        }
    });
    for (int i = n_edges + lane; i < a.E; i += 64) {   // unused edge slots read as no edge
        em[i] = 0;
        ep[i] = (_Float16)0.0f;
    }
    if (lane == 0) write_counts(a, b, n_edges, total, trunc, s_all, s_keep);
}

// The candidates of a wavefront's two positions, one half each (lane s of it owns slot s): m64 its legal-move word, pr the
// squares of it that promote, cnt its candidates and before those of the slots in front; total0 / total1 the two
// positions' (most: the larger, at most 32 ROUNDS).  A half's result does not depend on the other one.
template <bool FP32, int ROUNDS>
__device__ __forceinline__ void expand_pair(const KExpand& a, const Shared& sh, int b, bool ok, int s, int half, uint64_t m64, uint64_t pr, int cnt, int before,
                                            int total0, int total1, int total, int most) {
    const int rounds = (most + 31) >> 5;
    int16_t* const cc = sh.code;
    float* const add = sh.add;
    const size_t row = (size_t)b * 2048;
    float l[ROUNDS], e[ROUNDS];
    int code[ROUNDS];
    bool has[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        has[r] = 32 * r + s < total;
        l[r] = -INFINITY;
        code[r] = 0;
    }
    if (__ballot(pr != 0) == 0) {
        // the slot a candidate belongs to: the last one whose first index is not beyond it
        unsigned char* const owner = reinterpret_cast<unsigned char*>(sh.owner);
#pragma unroll
        for (int r = 0; r < ROUNDS; r += 4) sh.owner[8 * r + s] = 0;
        wave_lds_sync();
        if (cnt) owner[before] = (unsigned char)s;
        wave_lds_sync();
        int carry0 = 0, carry1 = 0;
        const int mlo = (int)(unsigned)m64, mhi = (int)(unsigned)(m64 >> 32);
#pragma unroll
        for (int r = 0; r < ROUNDS; r++)
            if (r < rounds) {
                const int own = max(half_scan_max(owner[32 * r + s]), half ? carry1 : carry0);
                carry0 = __builtin_amdgcn_readlane(own, 31);
                carry1 = __builtin_amdgcn_readlane(own, 63);
                const int src = 4 * (32 * half + own);
                const int k = 32 * r + s - __builtin_amdgcn_ds_bpermute(src, before);
                const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(src, mlo), hi = (unsigned)__builtin_amdgcn_ds_bpermute(src, mhi);
                if (has[r]) {
                    code[r] = own * 64 + kth_bit(lo, hi, k);
                    l[r] = logit<FP32>(a.policy, row + code[r]);
                }
            }
    } else {
        float lp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (pr) promotion_logs<FP32>(a.promo, (size_t)b * 32 + s, lp);
        int i = before;
        for (uint64_t m = m64; m; m &= m - 1) {
            const int sq = __builtin_ctzll(m), mv = s * 64 + sq;
            if ((pr >> sq) & 1) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    cc[i + k] = (int16_t)(mv | (k << PROMO_SHIFT));
                    add[i + k] = lp[k];
                }
                i += 4;
            } else {
                cc[i] = (int16_t)mv;
                add[i++] = 0.0f;
            }
        }
        wave_lds_sync();
#pragma unroll
        for (int r = 0; r < ROUNDS; r++)
            if (has[r]) {
                code[r] = cc[32 * r + s];
                l[r] = logit<FP32>(a.policy, row + (code[r] & 2047)) + add[32 * r + s];
            }
        wave_lds_sync();
    }
    float mx = l[0];
#pragma unroll
    for (int r = 1; r < ROUNDS; r++) mx = fmaxf(mx, l[r]);
    mx = half_max(mx);
    float sa = 0.0f;
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        e[r] = 0.0f;
        if (r < rounds) e[r] = has[r] ? __expf(l[r] - mx) : 0.0f;
        sa += e[r];
    }
    const float s_all = half_sum(sa);
    const bool trunc = total > a.E;
    int n_edges = total;
    float s_keep = s_all;
    int pos[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) pos[r] = 32 * r + s;
    if (most > a.E) {
        // T = ordered pattern of the E-th largest log-prior of each half (0: everything is kept)
        unsigned o[ROUNDS];
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) o[r] = has[r] ? ordered(l[r]) : 0u;
        // -- or any pattern that exactly E of its candidates reach, which ends the search for that half early
        unsigned T0 = 0, T1 = 0;
        bool found0 = total0 <= a.E, found1 = total1 <= a.E;
#pragma clang loop unroll(disable)
        for (int bit = 31; bit >= 0 && !(found0 && found1); bit--) {
            const unsigned cand = (half ? T1 : T0) | (1u << bit);
            int c0 = 0, c1 = 0;
#pragma unroll
            for (int r = 0; r < ROUNDS; r++)
                if (r < rounds) {
                    const unsigned long long v = __ballot(o[r] >= cand);
                    c0 += __popc((unsigned)v);
                    c1 += __popc((unsigned)(v >> 32));
                }
            if (!found0 && c0 >= a.E) T0 |= 1u << bit;
            if (!found1 && c1 >= a.E) T1 |= 1u << bit;
            found0 |= c0 == a.E;
            found1 |= c1 == a.E;
        }
        const unsigned T = half ? T1 : T0;
        int gt = 0;
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {
            const unsigned long long v = __ballot(o[r] > T);
            gt += __popc(half ? (unsigned)(v >> 32) : (unsigned)v);
        }
        const int need = a.E - gt;
        int ties = 0, kept = 0;
        float sk = 0.0f;
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {
            const bool eq = has[r] && o[r] == T;
            const unsigned long long eqb = __ballot(eq);
            has[r] = has[r] && (o[r] > T || (eq && ties + half_below(eqb, half) < need));
            ties += __popc(half ? (unsigned)(eqb >> 32) : (unsigned)eqb);
            const unsigned long long kb = __ballot(has[r]);
            pos[r] = kept + half_below(kb, half);
            kept += __popc(half ? (unsigned)(kb >> 32) : (unsigned)kb);
            sk += has[r] ? e[r] : 0.0f;
        }
        n_edges = kept;
        s_keep = half_sum(sk);
    }
    const float inv = 1.0f / s_keep;
    int16_t* const em = a.edge_move + (size_t)b * a.E;
    _Float16* const ep = a.edge_prior + (size_t)b * a.E;
    if (a.whole_rows) {
        // rows of whole 16-byte pieces: put together in LDS, unused slots (no edge) included
        _Float16* const pp = sh.prior;
        typedef int v4i __attribute__((ext_vector_type(4)));
        reinterpret_cast<v4i*>(cc)[s] = v4i{0, 0, 0, 0};
        reinterpret_cast<v4i*>(pp)[s] = v4i{0, 0, 0, 0};
        wave_lds_sync();
#pragma unroll
        for (int r = 0; r < ROUNDS; r++)
            if (r < rounds && has[r]) {
                cc[pos[r]] = (int16_t)code[r];
                pp[pos[r]] = (_Float16)(e[r] * inv);
            }
        wave_lds_sync();
        if (ok && s < a.E / 8) {
            reinterpret_cast<v4i*>(em)[s] = reinterpret_cast<const v4i*>(cc)[s];
            reinterpret_cast<v4i*>(ep)[s] = reinterpret_cast<const v4i*>(pp)[s];
        }
    } else {
#pragma unroll
        for (int r = 0; r < ROUNDS; r++)
            if (has[r]) {
                em[pos[r]] = (int16_t)code[r];
                ep[pos[r]] = (_Float16)(e[r] * inv);
            }
        if (ok)
            for (int i = n_edges + s; i < a.E; i += 32) {
                em[i] = 0;
                ep[i] = (_Float16)0.0f;
            }
    }
    if (ok && s == 0) write_counts(a, b, n_edges, total, trunc, s_all, s_keep);
}

// GENERATE: the legal-move words are made here, in a launch less.  Both rows of sixteen lanes of a half generate its position's moves, so that
// each lane has the word of a slot; with two positions instead of four to a wavefront that costs twice the instructions, which
// small launches, bound by the launch itself, do not notice: both as calls of their own 11.1 -> 6.8 us for 64 positions, 11.7 -> 7.1 for 4096, 12.1
// -> 9.6 for 8192, 13.7 -> 12.4 for 12000, but 17.0 -> 17.6 for 20000 and 40.4 -> 45.3 for 65536; behind an evaluation of 64 85.9 -> 84.0, and
// from 1000 on less than runs differ by (4096: 1415 and 1421, 12000: 4162 and 4158).
template <bool FP32, bool GENERATE>
__global__ __launch_bounds__(64 * EXPAND_WAVES) void expand_kernel(const KExpand a) {
    __shared__ bf::moves::Table table;
    static_assert(!GENERATE || EXPAND_WAVES == 4, "a wavefront a field of the table");
    if constexpr (GENERATE) bf::moves::fill(table);
    __shared__ __attribute__((aligned(16))) int16_t code_lds[EXPAND_WAVES][2][CAND_CAP];
    __shared__ __attribute__((aligned(16))) _Float16 prior_lds[EXPAND_WAVES][2][CAND_CAP];
    __shared__ float add_lds[EXPAND_WAVES][2][CAND_CAP];
    __shared__ unsigned owner_lds[EXPAND_WAVES][2][CAND_CAP / 4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, s = lane & 31, half = lane >> 5;
    const int j = 2 * (blockIdx.x * EXPAND_WAVES + wv) + half;
    // the half's position; a half without one has no candidates and stores nothing
    int b = j;
    bool ok = j < a.n;
    if (a.leaf_index) {
        ok = ok && j < *a.leaf_count;
        b = ok ? a.leaf_index[j] : 0;
        ok = ok && (unsigned)b < (unsigned)a.n;
    }
    if (ok && a.active) ok = a.active[b] != 0;
    if (!ok) b = 0;
    if (__ballot(ok) == 0) return;                       // no workgroup barrier below: a wave may leave

    const unsigned word = a.boards[(size_t)b * 32 + s];
    const int ctrl = a.control[b];
    uint64_t m64;
    if constexpr (GENERATE) {
        const bool black = ctrl < 0;
        const uint64_t legal = bf::moves::of_row(a.boards + (size_t)b * 32, black, lane, table, [&](bool attacked) {
            if (ok && s == 15) a.in_check[b] = attacked;
        });
        m64 = ok && (s >> 4) == (int)black ? legal : 0;
        if (ok) a.mask_out[(size_t)b * 32 + s] = m64;
    } else m64 = ok ? a.mask[(size_t)b * 32 + s] : 0;
    const bool pawn = ((word >> 11) & 1u) == 0 && ((word >> 6) & 7u) == PAWN;
    // last rank of the side to move: rank 7 (squares 56..63) for white, rank 0 for black
    uint64_t pr = pawn ? m64 & (ctrl < 0 ? 0xFFull : 0xFFull << 56) : 0;
    int cnt = __popcll(m64) + 3 * __popcll(pr);
    const int inc = half_scan_add(cnt);
    int before = inc - cnt;
    int total0 = __builtin_amdgcn_readlane(inc, 31), total1 = __builtin_amdgcn_readlane(inc, 63);
    int total = half ? total1 : total0, most = max(total0, total1);
    if (most > CAND_CAP) {
        // a position with more goes through the whole wavefront first and leaves an empty half behind; the other
        // half's goes on as it would beside any neighbour
        if constexpr (GENERATE) __threadfence();   // it reads the words back
        if (total0 > CAND_CAP) expand_many<FP32>(a, __builtin_amdgcn_readlane(b, 0), lane);
        if (total1 > CAND_CAP) expand_many<FP32>(a, __builtin_amdgcn_readlane(b, 32), lane);
        const bool many = total > CAND_CAP;
        ok = ok && !many;
        if (__ballot(ok) == 0) return;
        m64 = many ? 0 : m64;
        pr = many ? 0 : pr;
        cnt = many ? 0 : cnt;
        before = many ? 0 : before;
        total0 = total0 > CAND_CAP ? 0 : total0;
        total1 = total1 > CAND_CAP ? 0 : total1;
        total = half ? total1 : total0;
        most = max(total0, total1);
    }
    const Shared sh = {code_lds[wv][half], prior_lds[wv][half], add_lds[wv][half], owner_lds[wv][half]};
    if (most <= 32 * FEW_ROUNDS) expand_pair<FP32, FEW_ROUNDS>(a, sh, b, ok, s, half, m64, pr, cnt, before, total0, total1, total, most);
    else expand_pair<FP32, MOST_ROUNDS>(a, sh, b, ok, s, half, m64, pr, cnt, before, total0, total1, total, most);
}

}  // namespace

// Order-preserving compaction of the leaf flags.  A workgroup takes 16384 flags, sixteen per lane in one
// load; where they go in the list is the number of live flags in front of them, which every workgroup
// counts for itself (16 flags per lane and load again: 64 KiB in a microsecond or two), so no workgroup
// waits for another and nothing is kept between launches.  One workgroup going through all flags, a byte
// per lane and two barriers per 1024, took 41 us for 65536 flags, this 4.2 us (4096 flags: 10 us
// before, 3.2).  The counting grows with the square of the workgroups, so there are at most 256 of them, one per
// compute unit, which beyond 4 M flags take several runs of 16384 each: 2^24 flags take 0.16 ms, 2^28
// 3 ms (with a workgroup for every 16384: 0.77 and 251; one workgroup: 12 and 237).
constexpr int COMPACT_LANES = 1024, COMPACT_FLAGS = 16, COMPACT_GROUPS = 256;
constexpr int COMPACT_CHUNK = COMPACT_LANES * COMPACT_FLAGS;

// the high bit of every non-zero byte
__device__ __forceinline__ unsigned nonzero_bytes(unsigned x) { return (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u; }

// sixteen flags from `at` on (zero past the end) as a 16-bit mask
__device__ __forceinline__ unsigned flag_bits(const uint8_t* flags, long long at, long long n, bool aligned) {
    unsigned bits = 0;
    if (aligned && at + COMPACT_FLAGS <= n) {
        const uint4 v = *reinterpret_cast<const uint4*>(flags + at);
        const unsigned d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned h = nonzero_bytes(d[i]) >> 7;   // bits 0, 8, 16, 24
            bits |= ((h | h >> 7 | h >> 14 | h >> 21) & 15u) << (4 * i);
        }
    } else {
        for (int i = 0; i < COMPACT_FLAGS; i++)
            if (at + i < n && flags[at + i]) bits |= 1u << i;
    }
    return bits;
}

template <bool ONE_RUN>   // (the loop costs a launch of few flags 0.4 us)
__global__ __launch_bounds__(COMPACT_LANES) void compact_kernel(const uint8_t* flags, int n, int chunks_, int* leaf_index, int* leaf_count) {
    const int chunks = ONE_RUN ? 1 : chunks_;
    __shared__ int total[2][COMPACT_LANES / 64], ahead[COMPACT_LANES / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool aligned = ((uintptr_t)flags & 15) == 0;
    const long long first = (long long)blockIdx.x * chunks * COMPACT_CHUNK;   // this workgroup's flags: `chunks` runs of 16384
    int front = 0;
    if (aligned) {
#pragma unroll 4
        for (long long at = (long long)threadIdx.x * COMPACT_FLAGS; at < first; at += COMPACT_CHUNK) {
            const uint4 v = *reinterpret_cast<const uint4*>(flags + at);
            front += __popc(nonzero_bytes(v.x)) + __popc(nonzero_bytes(v.y)) + __popc(nonzero_bytes(v.z)) + __popc(nonzero_bytes(v.w));
        }
    } else {
#pragma unroll 1
        for (long long at = (long long)threadIdx.x * COMPACT_FLAGS; at < first; at += COMPACT_CHUNK) front += __popc(flag_bits(flags, at, n, false));
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) front += __shfl_xor(front, d);
    if (lane == 63) ahead[wave] = front;
    int base = 0;
    for (int c = 0; c < chunks; c++) {
        const long long run = first + (long long)c * COMPACT_CHUNK;
        if (!ONE_RUN && run >= n) break;
        const int mine = (int)run + (int)threadIdx.x * COMPACT_FLAGS;
        unsigned bits = flag_bits(flags, mine, n, aligned);
        const int cnt = __popc(bits);
        int inc = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d);
            if (lane >= d) inc += o;
        }
        if (lane == 63) total[c & 1][wave] = inc;
        __syncthreads();   // one a run: the totals of the run after the next are written behind the next one's
        int at = inc - cnt, all = 0;
#pragma unroll
        for (int w = 0; w < COMPACT_LANES / 64; w++) {
            base += c == 0 ? ahead[w] : 0;
            at += w < wave ? total[c & 1][w] : 0;
            all += total[c & 1][w];
        }
        at += base;
        for (; bits; bits &= bits - 1) leaf_index[at++] = mine + __builtin_ctz(bits);
        base += all;
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *leaf_count = base;
}

extern "C" int bf_compact_leaves(const uint8_t* flags, int64_t n, int32_t* leaf_index, int32_t* leaf_count, void* stream) {
    auto fail = [](int code, const char* msg) {
        bf::set_error(msg);
        return code;
    };
    if (!flags || !leaf_index || !leaf_count) return fail(BF_ERR_ARGUMENT, "flags/leaf_index/leaf_count must not be NULL");
    if (n < 1 || n > (1ll << 28)) return fail(BF_ERR_ARGUMENT, "n must be in [1, 2^28]");
    if (((uintptr_t)leaf_index & 3) || ((uintptr_t)leaf_count & 3)) return fail(BF_ERR_ARGUMENT, "leaf_index / leaf_count must be 4-byte aligned");
    const int runs = (int)((n + COMPACT_CHUNK - 1) / COMPACT_CHUNK), chunks = (runs + COMPACT_GROUPS - 1) / COMPACT_GROUPS;
    hipLaunchKernelGGL(chunks == 1 ? compact_kernel<true> : compact_kernel<false>, dim3((unsigned)((runs + chunks - 1) / chunks)), dim3(COMPACT_LANES), 0, (hipStream_t)stream,
                       flags, (int)n, chunks, leaf_index, leaf_count);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        char msg[256];
        snprintf(msg, sizeof(msg), "kernel launch failed: %s", hipGetErrorString(e));
        return fail(BF_ERR_LAUNCH, msg);
    }
    return BF_OK;
}

constexpr int CLEAR_MOST = 8, CLEAR_LANES = 256, CLEAR_PIECES = 4;   // sixteen bytes a piece
struct KClear {
    uint8_t* at[CLEAR_MOST];
    size_t bytes[CLEAR_MOST];
};
__global__ __launch_bounds__(CLEAR_LANES) void clear_kernel(const KClear k) {
    uint8_t* const to = k.at[blockIdx.y];
    const size_t bytes = k.bytes[blockIdx.y], whole = bytes / 16;
#pragma unroll
    for (int i = 0; i < CLEAR_PIECES; i++) {
        const size_t piece = ((size_t)blockIdx.x * CLEAR_PIECES + i) * CLEAR_LANES + threadIdx.x;
        if (piece < whole) reinterpret_cast<uint4*>(to)[piece] = uint4{0, 0, 0, 0};
        else if (piece == whole)
            for (size_t b = 16 * whole; b < bytes; b++) to[b] = 0;
    }
}

extern "C" int bf_clear(void* const* buffers, const size_t* bytes, int n, void* stream) {
    auto fail = [](int code, const char* msg) {
        bf::set_error(msg);
        return code;
    };
    if (!buffers || !bytes || n < 1 || n > CLEAR_MOST) return fail(BF_ERR_ARGUMENT, "buffers/bytes must not be NULL, n in [1, 8]");
    KClear k = {};
    size_t most = 0;
    for (int i = 0; i < n; i++) {
        if ((!buffers[i] && bytes[i]) || ((uintptr_t)buffers[i] & 15)) return fail(BF_ERR_ARGUMENT, "a buffer must be 16-byte aligned and not NULL");
        k.at[i] = static_cast<uint8_t*>(buffers[i]);
        k.bytes[i] = bytes[i];
        most = bytes[i] > most ? bytes[i] : most;
    }
    constexpr size_t per = 16 * CLEAR_LANES * CLEAR_PIECES;
    if (most >= (per << 31)) return fail(BF_ERR_ARGUMENT, "a buffer is too large");
    if (!most) return BF_OK;
    hipLaunchKernelGGL(clear_kernel, dim3((unsigned)(most / per + 1), n), dim3(CLEAR_LANES), 0, (hipStream_t)stream, k);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        char msg[256];
        snprintf(msg, sizeof(msg), "kernel launch failed: %s", hipGetErrorString(e));
        return fail(BF_ERR_LAUNCH, msg);
    }
    return BF_OK;
}

// bf_expand, and with in_check the move generation in front of it (a->mask is where its words go)
static int expand(const bf_expand_args* a, uint64_t* mask_out, uint8_t* in_check, void* stream) {
    auto fail = [](int code, const char* msg) {
        bf::set_error(msg);
        return code;
    };
    if (!a) return fail(BF_ERR_ARGUMENT, "args is NULL");
    if (a->n < 1 || a->n > (1ll << 28)) return fail(BF_ERR_ARGUMENT, "n must be in [1, 2^28]");
    if (a->max_edges < 1 || a->max_edges > 255) return fail(BF_ERR_ARGUMENT, "max_edges must be in [1, 255]");
    if (!a->policy || !a->promo || !a->mask || !a->boards || !a->control)
        return fail(BF_ERR_ARGUMENT, "policy/promo/mask/boards/control must not be NULL");
    if (!a->edge_move || !a->edge_prior || !a->n_edges) return fail(BF_ERR_ARGUMENT, "edge_move/edge_prior/n_edges must not be NULL");
    if (a->node_value && !a->value) return fail(BF_ERR_ARGUMENT, "node_value needs value");
    if (((uintptr_t)a->policy & 15) || ((uintptr_t)a->mask & 7) || ((uintptr_t)a->promo & 1))
        return fail(BF_ERR_ARGUMENT, "policy must be 16-byte and mask 8-byte aligned");
    KExpand k = {};
    k.mask_out = mask_out; k.in_check = in_check;
    k.policy = a->policy; k.promo = a->promo; k.value = a->value; k.mask = a->mask;
    if ((a->leaf_index == nullptr) != (a->leaf_count == nullptr)) return fail(BF_ERR_ARGUMENT, "leaf_index and leaf_count come together");
    if (a->leaf_index && a->active) return fail(BF_ERR_ARGUMENT, "a compacted leaf list replaces the active flags: pass one of them");
    k.boards = a->boards; k.control = a->control; k.active = a->active;
    k.leaf_index = a->leaf_index; k.leaf_count = a->leaf_count;
    k.n = (int)a->n; k.E = a->max_edges; k.logits_fp32 = a->logits_fp32 ? 1 : 0;
    k.edge_move = a->edge_move; k.edge_prior = reinterpret_cast<_Float16*>(a->edge_prior);
    k.n_edges = a->n_edges; k.count = a->count; k.dropped = a->dropped;
    k.node_value = reinterpret_cast<_Float16*>(a->node_value);
    k.whole_rows = k.E % 8 == 0 && k.E <= CAND_CAP && (((uintptr_t)k.edge_move | (uintptr_t)k.edge_prior) & 15) == 0;
    const dim3 grid((k.n + 2 * EXPAND_WAVES - 1) / (2 * EXPAND_WAVES)), block(64 * EXPAND_WAVES);
    void (*const kernel)(KExpand) = mask_out ? (k.logits_fp32 ? &expand_kernel<true, true> : &expand_kernel<false, true>)
                                             : (k.logits_fp32 ? &expand_kernel<true, false> : &expand_kernel<false, false>);
    hipLaunchKernelGGL(kernel, grid, block, 0, (hipStream_t)stream, k);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        char msg[256];
        snprintf(msg, sizeof(msg), "kernel launch failed: %s", hipGetErrorString(e));
        return fail(BF_ERR_LAUNCH, msg);
    }
    return BF_OK;
}

extern "C" int bf_expand(const bf_expand_args* a, void* stream) { return expand(a, nullptr, nullptr, stream); }

extern "C" int bf_movegen_expand(const bf_expand_args* args, uint64_t* mask, uint8_t* in_check, void* stream) {
    auto fail = [](int code, const char* msg) {
        bf::set_error(msg);
        return code;
    };
    if (!args || !mask || !in_check) return fail(BF_ERR_ARGUMENT, "args/mask/in_check must not be NULL");
    if (args->mask || args->active || args->leaf_index || args->leaf_count)
        return fail(BF_ERR_ARGUMENT, "bf_movegen_expand generates and expands every position: no mask, flags or leaf list");
    if (((uintptr_t)args->boards & 1) || ((uintptr_t)args->control & 1)) return fail(BF_ERR_ARGUMENT, "boards and control must be 2-byte aligned");
    bf_expand_args a = *args;
    a.mask = mask;
    return expand(&a, mask, in_check, stream);
}
