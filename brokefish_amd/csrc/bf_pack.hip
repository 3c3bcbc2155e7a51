// Weights of a network, as they lie in a trainer's fp32 parameters on the GPU, into the two blobs the
// one-position-per-workgroup kernels read (board_wstream / board_fparams, layout at the end of
// include/brokefish_hip.h): quantised per 128-row block (int8: over the whole reduction, reference
// brokefish/nn/quant.py:263-278; e4m3: per 256-deep k-chunk, quant.py:208-224) and laid out in the
// kernels' consumption order.  brokefish_amd/hip_impl.py pack_network_board is the same function in
// numpy and its checker; the bytes are identical (IEEE divisions, round to nearest even).
//
// Two launches per group of layers, both bound by launch latency and one pass over the parameters
// (25 MB for the 8-layer network): the largest magnitude of every 32 x 256 weight tile, then one
// workgroup per tile that takes its block's scale from the tile maxima, quantises and stores the
// tile's 8 KiB block where it belongs -- no atomics and nothing to clear, and 768 workgroups for the
// 8-layer network where one workgroup per scale block would be 144.  Packing on the host took 39 ms
// for that network and copied the parameters there and the blobs back; these two launches take 13 us.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "bf_device.hip.h"

namespace bf {
namespace pack {

constexpr int GROUP_LAYERS = 16;   // layers per launch: their pointers travel in the kernel arguments (1.5 KiB)

struct LayerGroup {
    bf_layer_weights w[GROUP_LAYERS];
    bf_global_weights g;
    uint8_t* wstream;
    float* fparams;
    float* amax;          // [n_layers][TILES], the largest magnitude of every weight tile
    int l0, nl, n_layers, n_value, fp8;
};

// A layer's weight tiles in the order QKV (3 NT row tiles x KC chunks), out-projection (NT x KC), first
// (4 NT x KC) and second (NT x KCF) feed-forward matrix.
template <int DM>
struct Tiles : Layout<DM> {
    typedef Layout<DM> L;
    static constexpr int QKV = 0, OUT = 3 * L::NT * L::KC, FF1 = OUT + L::NT * L::KC, FF2 = FF1 + 4 * L::NT * L::KC,
                         TILES = FF2 + L::NT * L::KCF;
    static_assert(TILES == 4 * L::BPW, "a layer's blocks");
};

struct TileOf {
    const float* w;       // the matrix, [rows, k]
    int k, first, n, c, chunks, part;   // row length; first tile of the matrix; row tile, k-chunk; chunks per row tile; which matrix
};

template <int DM>
__device__ __forceinline__ TileOf tile_of(const bf_layer_weights& w, int i) {
    typedef Tiles<DM> C;
    if (i < C::OUT) return {w.in_proj_w, DM, C::QKV, i / C::KC, i % C::KC, C::KC, 0};
    if (i < C::FF1) return {w.out_proj_w, DM, C::OUT, (i - C::OUT) / C::KC, (i - C::OUT) % C::KC, C::KC, 1};
    if (i < C::FF2) return {w.linear1_w, DM, C::FF1, (i - C::FF1) / C::KC, (i - C::FF1) % C::KC, C::KC, 2};
    return {w.linear2_w, C::F, C::FF2, (i - C::FF2) / C::KCF, (i - C::FF2) % C::KCF, C::KCF, 3};
}

// the scale of the 128-row block that row tile n of a matrix belongs to (e4m3: at k-chunk c)
__device__ __forceinline__ float block_scale(const float* amax, int first, int n, int c, int chunks, bool fp8) {
    float m = 0.0f;
    const float* p = amax + first + (n & ~3) * chunks;
    for (int i = 0; i < 4 * chunks; i++)
        if (!fp8 || i % chunks == c) m = __builtin_fmaxf(m, p[i]);
    return m > 0.0f ? m / (fp8 ? 8.0f : 127.0f) : 1.0f;
}

// the same, a tile's maximum per lane (at most 32: eight chunks of four tiles) instead of one after the other, with the tile's
// own values under way: the packing launch 9.1 -> 8.2 us
__device__ __forceinline__ float block_scale_of_lanes(const float* amax, int first, int n, int c, int chunks, bool fp8, int lane) {
    float m = 0.0f;
    if (lane < 4 * chunks && (!fp8 || lane % chunks == c)) m = __builtin_fmaxf(m, amax[first + (n & ~3) * chunks + lane]);
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, d));
    m = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(m)));
    return m > 0.0f ? m / (fp8 ? 8.0f : 127.0f) : 1.0f;
}

template <int DM>
__global__ __launch_bounds__(256) void amax_kernel(const LayerGroup a) {
    typedef Tiles<DM> C;
    const int l = (int)blockIdx.x / C::TILES, i = (int)blockIdx.x % C::TILES;
    const TileOf t = tile_of<DM>(a.w[l], i);
    // 64 lanes read one row's 1 KiB, a wave eight of the tile's 32 rows
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float* src = t.w + (size_t)(32 * t.n + wave) * t.k + 256 * t.c + 4 * lane;
    float m = 0.0f;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const v4f v = ldg4(src + (size_t)(4 * r) * t.k);
#pragma unroll
        for (int j = 0; j < 4; j++) m = __builtin_fmaxf(m, __builtin_fabsf(v[j]));
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, d));
    __shared__ float part[4];
    if (lane == 0) part[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        a.amax[(size_t)(a.l0 + l) * C::TILES + i] =
            __builtin_fmaxf(__builtin_fmaxf(part[0], part[1]), __builtin_fmaxf(part[2], part[3]));
}

template <int DM>
__device__ __forceinline__ void pack_tile(const LayerGroup& a, int l, int i) {
    typedef Tiles<DM> C;
    const int lane = threadIdx.x & 63, s = threadIdx.x >> 6, o = lane & 31, g = lane >> 5;
    const TileOf t = tile_of<DM>(a.w[l], i);
    // fragment s of the block: this lane's 16 operand bytes
    const float* src = t.w + (size_t)(32 * t.n + o) * t.k + 256 * t.c + 32 * s + 4 * g;
    v4f in[4];
#pragma unroll
    for (int j = 0; j < 4; j++) in[j] = ldg4(src + 8 * j);
    const float sw = block_scale_of_lanes(a.amax + (size_t)(a.l0 + l) * C::TILES, t.first, t.n, t.c, t.chunks, a.fp8, lane);
    v4i out;
    int sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float q[4];
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = in[j][k] / sw;
        if (a.fp8) {
#pragma unroll
            for (int k = 0; k < 4; k++) q[k] = __builtin_fminf(__builtin_fmaxf(q[k], -448.0f), 448.0f);
            int w = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
            out[j] = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], w, true);
        } else {
            unsigned w = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int b = (int)__builtin_fminf(__builtin_fmaxf(__builtin_rintf(q[k]), -127.0f), 127.0f);
                sum += b;
                w |= (unsigned)(b & 255) << (8 * k);
            }
            out[j] = (int)w;
        }
    }
    // where the kernels' wave (quarter) `wq` reads the block in its stream of this layer
    int wq, at;
    constexpr int SSTR = 4 * C::KC + 2 * C::TW, BASE = 4 * C::TW * C::KC;
    if (t.part == 0) {
        const int n = t.n % C::NT;
        wq = n / C::TW;
        at = (3 * (n % C::TW) + t.n / C::NT) * C::KC + t.c;
    } else if (t.part == 1) {
        wq = t.n / C::TW;
        at = (3 * C::TW + t.n % C::TW) * C::KC + t.c;
    } else if (t.part == 2) {
        wq = (t.n % 16) / 4;
        at = BASE + (t.n / 16) * SSTR + (t.n % 4) * C::KC + t.c;
    } else {
        wq = t.n / C::TW;
        at = BASE + (t.c / 2) * SSTR + 4 * C::KC + (t.c % 2) * C::TW + t.n % C::TW;
    }
    const size_t blk = (size_t)wq * ((size_t)a.n_layers * C::BPW + C::HB + 1) + (size_t)(a.l0 + l) * C::BPW + at;
    *reinterpret_cast<v4i*>(a.wstream + blk * BLOCK + s * FRAG + lane * 16) = out;
    // 128 * the sum of the chunk's weights per row, the offset of the unsigned hidden operand
    if (t.part == 3) {
        __shared__ int rows[8][32];
        sum += __shfl_xor(sum, 32);
        if (g == 0) rows[s][o] = sum;
        __syncthreads();
        if (threadIdx.x < 32) {
            int all = 0;
#pragma unroll
            for (int f = 0; f < 8; f++) all += rows[f][threadIdx.x];
            float* const p = a.fparams + ((size_t)wq * a.n_layers + a.l0 + l) * C::PW_FLOATS + C::A_FLOATS;
            p[C::B_WSUM + t.c * C::CW + 32 * (t.n % C::TW) + threadIdx.x] = __int_as_float(a.fp8 ? 0 : 128 * all);
        }
    }
}

// the side parameters of quarter wq of a layer (all but the row sums, which the tiles write)
template <int DM>
__device__ __forceinline__ void pack_params(const LayerGroup& a, int l, int wq) {
    typedef Tiles<DM> C;
    const bf_layer_weights& w = a.w[l];
    const float* const amax = a.amax + (size_t)(a.l0 + l) * C::TILES;
    float* const p = a.fparams + ((size_t)wq * a.n_layers + a.l0 + l) * C::PW_FLOATS;
    const bool fp8 = a.fp8;
    for (int i = threadIdx.x; i < C::A_FLOATS + C::B_WSUM; i += 512) {
        float v = 0.0f;
        if (i < C::A_SW) {
            const int part = i / C::CW, ch_ = C::CW * wq + i % C::CW;
            v = part == 0 ? w.norm1_w[ch_] : part == 1 ? w.norm1_b[ch_] : part == 5 ? w.out_proj_b[ch_]
                                                                                    : w.in_proj_b[(part - 2) * DM + ch_];
        } else if (i < C::A_FLOATS) {
            const int j = i - C::A_SW, part = j / C::TW, n = C::TW * wq + j % C::TW;
            if (part < 3) v = block_scale(amax, C::QKV, part * C::NT + n, 0, C::KC, fp8);
            else if (part == 3) v = block_scale(amax, C::OUT, n, 0, C::KC, fp8);
        } else {
            const int j = i - C::A_FLOATS;
            if (j < C::B_SW) {
                const int ch_ = C::CW * wq + j % C::CW, part = j / C::CW;
                v = part == 0 ? w.norm2_w[ch_] : part == 1 ? w.norm2_b[ch_] : w.linear2_b[ch_];
            } else if (j < C::B_LDS_FLOATS) {
                const int k = j - C::B_SW;
                if (k < 16) {
                    const int st = k / 4, n = 16 * st + 4 * wq + k % 4;
                    if (st < C::STEPS) v = block_scale(amax, C::FF1, n, 0, C::KC, fp8);
                } else if (fp8) {
                    const int n = (k - 16) / C::KCF, c = (k - 16) % C::KCF;
                    if (n < C::TW) v = block_scale(amax, C::FF2, C::TW * wq + n, c, C::KCF, true);
                } else if (k - 16 < C::TW) {
                    v = block_scale(amax, C::FF2, C::TW * wq + k - 16, 0, C::KCF, false);
                }
            } else {
                const int k = j - C::B_BFF1;
                v = w.linear1_b[512 * (k / 128) + 128 * wq + k % 128];
            }
        }
        p[i] = v;
    }
}

// block hb of the head tile of quarter wq ([policy; promo; value; zeros], rows 32 wq .. 32 wq + 31), or the
// block of zeros behind it
template <int DM>
__device__ __forceinline__ void pack_head(const LayerGroup& a, int wq, int hb) {
    typedef Tiles<DM> C;
    const int lane = threadIdx.x & 63, f = 8 * hb + (threadIdx.x >> 6), o = lane & 31, g = lane >> 5;
    const int row = 32 * wq + o, col = 32 * (f / 4) + 8 * (f % 4) + 4 * g;
    v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (hb < C::HB) {
        const float* src = row < BF_POLICY                          ? a.g.policy + (size_t)row * DM
                           : row < BF_POLICY + BF_PROMO             ? a.g.promo + (size_t)(row - BF_POLICY) * DM
                           : row < BF_POLICY + BF_PROMO + a.n_value ? a.g.value + (size_t)(row - BF_POLICY - BF_PROMO) * DM
                                                                    : nullptr;
        if (src) v = ldg4(src + col);
    }
    const size_t blk = (size_t)wq * ((size_t)a.n_layers * C::BPW + C::HB + 1) + (size_t)a.n_layers * C::BPW + hb;
    *reinterpret_cast<v4f*>(a.wstream + blk * BLOCK + (threadIdx.x >> 6) * FRAG + lane * 16) = v;
}

constexpr int GLOBAL_ROWS = 64 + 12 + 4 + 101 + 3 + 2;   // embedding tables and the final norm, in rows of the width

template <int DM>
__device__ __forceinline__ void pack_global(const LayerGroup& a, int first_row) {
    typedef Tiles<DM> C;
    float* const dst = a.fparams + (size_t)4 * a.n_layers * C::PW_FLOATS;
    for (int i = threadIdx.x; i < 8 * DM; i += 512) {
        int r = first_row + i / DM;
        const int c = i % DM;
        if (r >= GLOBAL_ROWS) return;
        float* const d = dst + (size_t)r * DM + c;
        const float* src = a.g.emb_square;
        if (r >= 64) { r -= 64; src = a.g.emb_type_special;
            if (r >= 12) { r -= 12; src = a.g.emb_color_turn;
                if (r >= 4) { r -= 4; src = a.g.emb_clock;
                    if (r >= 101) { r -= 101; src = a.g.emb_rep;
                        if (r >= 3) { r -= 3; src = r ? a.g.norm_f_b : a.g.norm_f_w; r = 0; } } } } }
        *d = src[(size_t)r * DM + c];
    }
}

template <int DM>
constexpr int globals_grid() { return 4 * (Layout<DM>::HB + 1) + (GLOBAL_ROWS + 7) / 8; }

template <int DM>
__global__ __launch_bounds__(512) void pack_kernel(const LayerGroup a) {
    typedef Tiles<DM> C;
    int i = (int)blockIdx.x;
    if (i < a.nl * C::TILES) return pack_tile<DM>(a, i / C::TILES, i % C::TILES);
    i -= a.nl * C::TILES;
    if (i < 4 * a.nl) return pack_params<DM>(a, i / 4, i % 4);
    i -= 4 * a.nl;   // the first group's launch also carries what does not belong to a layer
    if (i < 4 * (C::HB + 1)) return pack_head<DM>(a, i / (C::HB + 1), i % (C::HB + 1));
    pack_global<DM>(a, 8 * (i - 4 * (C::HB + 1)));
}

template <int DM>
hipError_t launch(LayerGroup& a, const bf_layer_weights* layers, hipStream_t stream) {
    typedef Tiles<DM> C;
    for (a.l0 = 0; a.l0 < a.n_layers; a.l0 += GROUP_LAYERS) {
        a.nl = a.n_layers - a.l0 < GROUP_LAYERS ? a.n_layers - a.l0 : GROUP_LAYERS;
        for (int l = 0; l < a.nl; l++) a.w[l] = layers[a.l0 + l];
        hipLaunchKernelGGL(amax_kernel<DM>, dim3(a.nl * C::TILES), dim3(256), 0, stream, a);
        const int grid = a.nl * (C::TILES + 4) + (a.l0 == 0 ? globals_grid<DM>() : 0);
        hipLaunchKernelGGL(pack_kernel<DM>, dim3(grid), dim3(512), 0, stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ---- the weight fingerprint ------------------------------------------------------------------------
// sum over parameters i of (i + 1) * sum_j f_j * (j % 9973 + 1), i and j counted from 0 and 1 (reference
// brokefish/train/sync.py:34-49), in float64.  One workgroup per 8192 elements leaves its partial sum, a
// second launch of one workgroup adds the partials in a fixed order: the same bits for the same
// weights every time.  Some eight launches and a host wait per parameter (106 of them for the 8-layer
// network) were 4 ms; these two launches take 12 us.
constexpr int FP_CHUNK = 8192, FP_GROUP = 192;   // elements per workgroup; parameters per launch (3 KiB of arguments)

struct FpGroup {
    const float* p[FP_GROUP];
    int before[FP_GROUP + 1];   // workgroups of the parameters in front
    int numel[FP_GROUP];
    int n, first;
    double* partial;
};

__device__ __forceinline__ double block_sum(double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
    __shared__ double part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    return (part[0] + part[1]) + (part[2] + part[3]);
}

// Bound by the latency of its loads: a thread asks for all its elements before it uses the first (eight at a time, each
// behind a check of its own: 14.5 us for the 8-layer network's 25 MB, 8.4 now; the second launch likewise, 4.0 us, 3.3).
__global__ __launch_bounds__(256) void fingerprint_kernel(const FpGroup a) {
    // the parameter this workgroup's elements belong to: the last one with no more workgroups in front (`before` rises)
    int lo = -1;
#pragma unroll
    for (int i = 0; i < FP_GROUP; i += 64) {
        const int k = i + (threadIdx.x & 63);
        lo += __builtin_popcountll(__ballot(k < a.n && a.before[k] <= (int)blockIdx.x));
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    const int at = ((int)blockIdx.x - a.before[lo]) * FP_CHUNK, end = a.numel[lo] - at;
    const float* const p = a.p[lo] + at;
    const double scale = (double)(a.first + lo + 1);
    constexpr int EACH = FP_CHUNK / 256;
    float v[EACH];
    if (end >= FP_CHUNK) {
#pragma unroll
        for (int j = 0; j < EACH; j++) v[j] = p[threadIdx.x + 256 * j];
    } else {
#pragma unroll
        for (int j = 0; j < EACH; j++) v[j] = (int)threadIdx.x + 256 * j < end ? p[threadIdx.x + 256 * j] : 0.0f;
    }
    double s = 0.0;
    unsigned weight = (unsigned)(at + (int)threadIdx.x + 1) % 9973u;
#pragma unroll
    for (int j = 0; j < EACH; j++) {
        s += (scale * (double)v[j]) * (double)(weight + 1u);
        weight += 256u;
        weight = weight >= 9973u ? weight - 9973u : weight;
    }
    s = block_sum(s);
    if (threadIdx.x == 0) a.partial[blockIdx.x] = s;
}

__global__ __launch_bounds__(256) void fingerprint_sum_kernel(const double* partial, int n, double* out) {
    double s = 0.0;
    for (int i0 = threadIdx.x; i0 < n; i0 += 256 * 8) {
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = i0 + 256 * j < n ? partial[i0 + 256 * j] : 0.0;
#pragma unroll
        for (int j = 0; j < 8; j++) s += v[j];
    }
    s = block_sum(s);
    if (threadIdx.x == 0) *out = s;
}

static int fail(int code, const char* msg) {
    set_error(msg);
    return code;
}

}  // namespace pack
}  // namespace bf

extern "C" size_t bf_pack_scratch_floats(const bf_shape* s) {
    if (bf_board_wstream_bytes(s) == 0) return 0;
    return (size_t)s->n_layers * 4 * (s->d_model == 256 ? bf::Layout<256>::BPW : bf::Layout<512>::BPW);
}

extern "C" int bf_pack_board(const bf_shape* s, int quant, const bf_layer_weights* layers, const bf_global_weights* g,
                             uint8_t* board_wstream, float* board_fparams, float* scratch, void* stream) {
    using bf::pack::fail;
    if (!s || bf_board_wstream_bytes(s) == 0) return fail(BF_ERR_UNSUPPORTED, "bf_pack_board: unsupported network shape");
    if (quant != BF_QUANT_INT8 && !(quant == BF_QUANT_E4M3 && s->d_model == 256))
        return fail(BF_ERR_UNSUPPORTED, "bf_pack_board: int8, or e4m3 for the 256-wide network");
    if (!layers || !g || !board_wstream || !board_fparams || !scratch)
        return fail(BF_ERR_ARGUMENT, "bf_pack_board: no pointer may be NULL");
    uintptr_t low = (uintptr_t)board_wstream | (uintptr_t)board_fparams;
    bool null = false;
    auto take = [&](const float* const* p, size_t count) {
        for (size_t i = 0; i < count; i++) {
            low |= (uintptr_t)p[i];
            null |= p[i] == nullptr;
        }
    };
    static_assert(sizeof(bf_layer_weights) == 12 * sizeof(float*) && sizeof(bf_global_weights) == 10 * sizeof(float*), "pointers only");
    take(reinterpret_cast<const float* const*>(layers), (size_t)12 * s->n_layers);
    take(reinterpret_cast<const float* const*>(g), 10);
    if (null || (low & 15) || ((uintptr_t)scratch & 3)) return fail(BF_ERR_ARGUMENT, "bf_pack_board: every parameter must be given, 16-byte aligned");
    if (!bf::device_is_gfx950()) return BF_ERR_DEVICE;
    bf::pack::LayerGroup a;
    a.g = *g;
    a.wstream = board_wstream;
    a.fparams = board_fparams;
    a.amax = scratch;
    a.n_layers = s->n_layers;
    a.n_value = s->n_value;
    a.fp8 = quant == BF_QUANT_E4M3;
    const hipError_t e = s->d_model == 256 ? bf::pack::launch<256>(a, layers, (hipStream_t)stream)
                                           : bf::pack::launch<512>(a, layers, (hipStream_t)stream);
    return e == hipSuccess ? BF_OK : fail(BF_ERR_LAUNCH, hipGetErrorString(e));
}

extern "C" int64_t bf_fingerprint_partials(const int64_t* numel, int n) {
    int64_t c = 0;
    for (int i = 0; i < n; i++) c += (numel[i] + bf::pack::FP_CHUNK - 1) / bf::pack::FP_CHUNK;
    return c;
}

extern "C" int bf_fingerprint(const float* const* params, const int64_t* numel, int n, double* partials, double* out, void* stream) {
    using bf::pack::fail;
    if (!params || !numel || !partials || !out || n < 1) return fail(BF_ERR_ARGUMENT, "bf_fingerprint: no pointer may be NULL, n >= 1");
    int64_t all = 0;
    for (int i = 0; i < n; i++) {
        if (!params[i] || ((uintptr_t)params[i] & 3) || numel[i] < 1 || numel[i] > (1 << 30))
            return fail(BF_ERR_ARGUMENT, "bf_fingerprint: a parameter is a non-NULL fp32 array of 1 to 2^30 elements");
        all += (numel[i] + bf::pack::FP_CHUNK - 1) / bf::pack::FP_CHUNK;
    }
    if (all > (1 << 30)) return fail(BF_ERR_ARGUMENT, "bf_fingerprint: too many elements");
    if (!bf::device_is_gfx950()) return BF_ERR_DEVICE;
    int64_t done = 0;
    for (int i0 = 0; i0 < n; i0 += bf::pack::FP_GROUP) {
        bf::pack::FpGroup a;
        a.n = n - i0 < bf::pack::FP_GROUP ? n - i0 : bf::pack::FP_GROUP;
        a.first = i0;
        a.partial = partials + done;
        a.before[0] = 0;
        for (int i = 0; i < a.n; i++) {
            a.p[i] = params[i0 + i];
            a.numel[i] = (int)numel[i0 + i];
            a.before[i + 1] = a.before[i] + (int)((numel[i0 + i] + bf::pack::FP_CHUNK - 1) / bf::pack::FP_CHUNK);
        }
        hipLaunchKernelGGL(bf::pack::fingerprint_kernel, dim3(a.before[a.n]), dim3(256), 0, (hipStream_t)stream, a);
        done += a.before[a.n];
    }
    hipLaunchKernelGGL(bf::pack::fingerprint_sum_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, partials, (int)done, out);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? BF_OK : fail(BF_ERR_LAUNCH, hipGetErrorString(e));
}
