// Host side of the evaluator library: the C-ABI of include/brokefish_hip.h.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <atomic>
#include <cstring>
#include <mutex>

#include "bf_args.h"



static thread_local char g_err[512] = "";

static int fail(int code, const char* msg) {
    snprintf(g_err, sizeof(g_err), "%s", msg);
    return code;
}

void bf::set_error(const char* msg) { snprintf(g_err, sizeof(g_err), "%s", msg); }

static bool shape_ok(const bf_shape* s) {   // the four-positions-per-workgroup kernel
    return s && s->d_model == bf::D && s->d_ff == bf::F && s->n_heads == bf::NH && s->n_layers >= 1 &&
           (s->n_value == 1 || s->n_value == 3);
}

static bool shape512(const bf_shape* s) {
    return s && s->d_model == 512 && s->d_ff == 2048 && s->n_heads == 16 && s->n_layers >= 1 &&
           (s->n_value == 1 || s->n_value == 3);
}

static bool board_shape_ok(const bf_shape* s) { return shape_ok(s) || shape512(s); }

// AUTO runs one workgroup of eight wavefronts per compute unit (lowest latency per position) up
// to this many positions, which is one per compute unit of an MI355X; above it, the forms built
// for throughput, with two positions per workgroup.
static const int64_t kBoardMaxN = 256;

template <int DM>
static size_t board_wstream_bytes(int n_layers) {
    typedef bf::Layout<DM> L;
    return (size_t)4 * ((size_t)n_layers * L::BPW + L::HB + 1) * bf::BLOCK;
}
template <int DM>
static size_t board_fparams_floats(int n_layers) {
    typedef bf::Layout<DM> L;
    return (size_t)4 * n_layers * L::PW_FLOATS + L::GLOBAL_FLOATS;
}

// Whether the kernels that reach their weights by 32-bit offsets carry a network of this depth: DUO, its one-position form and
// the 512-wide one with two positions, from the start of a quarter's stream (10,922 layers; 512 wide 2,730); the team form
// from the start of all four (2,730; 682).  Deeper networks stay on BOARD, TWIN and, 512 wide, OCTO.
static bool offsets_reach(const bf_shape* s, int quarters) {
    return bf_board_wstream_bytes(s) / 4 * quarters <= 0x7fffffff;
}

extern "C" size_t bf_board_wstream_bytes(const bf_shape* s) {
    if (shape_ok(s)) return board_wstream_bytes<256>(s->n_layers);
    if (shape512(s)) return board_wstream_bytes<512>(s->n_layers);
    return 0;
}

extern "C" size_t bf_board_fparams_floats(const bf_shape* s) {
    if (shape_ok(s)) return board_fparams_floats<256>(s->n_layers);
    if (shape512(s)) return board_fparams_floats<512>(s->n_layers);
    return 0;
}

extern "C" int64_t bf_board_max_n(void) { return kBoardMaxN; }

extern "C" uint64_t bf_abi_tag(void) { return BF_ABI_TAG; }

extern "C" size_t bf_wstream_bytes(const bf_shape* s) {
    if (!shape_ok(s)) return 0;
    return ((size_t)s->n_layers * bf::LAYER_GROUPS + bf::HEAD_GROUPS) * bf::GROUP;
}

extern "C" size_t bf_fparams_floats(const bf_shape* s) {
    if (!shape_ok(s)) return 0;
    return (size_t)s->n_layers * bf::PARAM_FLOATS + bf::GLOBAL_FLOATS;
}

extern "C" size_t bf_workspace_bytes(const bf_shape* s, int64_t n) {
    if (!shape_ok(s) || n < 1) return 0;
    const size_t slots = (size_t)((n + bf::WAVES - 1) / bf::WAVES) * bf::WAVES;
    return slots * bf::T * bf::D * sizeof(float);
}

extern "C" size_t bf_team_workspace_bytes(const bf_shape* s) {
    if (!board_shape_ok(s)) return 0;
    return bf::team_positions(s->d_model, true) * bf::team_slot_bytes(s->d_model);
}

extern "C" size_t bf_team_position_bytes(const bf_shape* s) { return board_shape_ok(s) ? bf::team_slot_bytes(s->d_model) : 0; }

extern "C" int bf_team_gave_up(void) { return bf::team_gave_up() ? 1 : 0; }

extern "C" size_t bf_layer_stride_floats(const bf_shape* s) {
    if (!shape_ok(s)) return 0;
    return bf::PARAM_FLOATS;
}

extern "C" void bf_int8_q_max(double* s8, double* u8) {
    if (s8) *s8 = 127.0;
    if (u8) *u8 = 255.0;
}

extern "C" double bf_fp8_q_max(void) { return 8.0; }

extern "C" const char* bf_last_error(void) { return g_err; }

// The kernel these arguments ask for, or whose launches they are (enum bf_kernel), or a negative status.
static int choose_kernel(const bf_eval_args* a) {
    if (!a) return fail(BF_ERR_ARGUMENT, "args is NULL");
    if (!board_shape_ok(&a->shape))
        return fail(BF_ERR_UNSUPPORTED,
                    "unsupported network shape: this build carries d_model=256/n_heads=8/d_ff=1024 and "
                    "d_model=512/n_heads=16/d_ff=2048, n_layers>=1, n_value in {1,3}");
    if (a->quant != BF_QUANT_INT8 && a->quant != BF_QUANT_E4M3)
        return fail(BF_ERR_ARGUMENT, "quant must be BF_QUANT_INT8 or BF_QUANT_E4M3");
    const bool have_quad = a->wstream && a->fparams, have_board = a->board_wstream && a->board_fparams;
    const bool quad_can = shape_ok(&a->shape) && have_quad;
    // the board blobs are packed for one format; the 512-wide network runs int8 only
    const bool board_can = have_board && (a->quant == BF_QUANT_INT8 || shape_ok(&a->shape));
    const bool twin_can = have_board && shape_ok(&a->shape);
    const bool reach = offsets_reach(&a->shape, 1);
    const bool octo_can = board_can && (reach || shape512(&a->shape));   // the same networks and formats as BOARD
    const bool duo_can = twin_can && reach;                              // the 256-wide network, both formats
    switch (a->kernel) {
    case BF_KERNEL_QUAD:
        if (!quad_can) return fail(BF_ERR_UNSUPPORTED, "the four-positions-per-workgroup kernel needs the 256-wide network and wstream/fparams");
        return BF_KERNEL_QUAD;
    case BF_KERNEL_BOARD:
        if (!board_can) return fail(BF_ERR_UNSUPPORTED, "the one-position-per-workgroup kernel needs board_wstream/board_fparams (512-wide network: the int8 format)");
        return BF_KERNEL_BOARD;
    case BF_KERNEL_TWIN:
        if (!twin_can)
            return fail(BF_ERR_UNSUPPORTED, "the two-workgroups-per-compute-unit kernel needs the 256-wide network and board_wstream/board_fparams");
        return BF_KERNEL_TWIN;
    case BF_KERNEL_OCTO:
        if (!octo_can)
            return fail(BF_ERR_UNSUPPORTED, "the eight-wavefronts-per-position kernel needs board_wstream/board_fparams (512-wide network: the int8 format; 256-wide: at most 10922 layers)");
        return BF_KERNEL_OCTO;
    case BF_KERNEL_DUO:
        if (!duo_can)
            return fail(BF_ERR_UNSUPPORTED, "the two-positions-per-workgroup kernel needs the 256-wide network, of at most 10922 layers, and board_wstream/board_fparams");
        return BF_KERNEL_DUO;
    case BF_KERNEL_AUTO:
        // above one position per compute unit: two positions per workgroup (int8: 5 to 8 % faster than TWIN from 512
        // positions up and half its L2 traffic).  For e4m3 the answer is still TWIN, what AUTO ran before the two-position
        // kernel overtook it; run_kernel() gives those launches to DUO.
        if (octo_can) return (twin_can && a->n > kBoardMaxN) ? (a->quant == BF_QUANT_INT8 ? BF_KERNEL_DUO : BF_KERNEL_TWIN) : BF_KERNEL_OCTO;
        if (board_can) return a->n > kBoardMaxN ? BF_KERNEL_TWIN : BF_KERNEL_BOARD;   // too deep for those
        if (quad_can) return BF_KERNEL_QUAD;
        return fail(BF_ERR_ARGUMENT, shape512(&a->shape)
                        ? "the 512-wide network runs on the one-position-per-workgroup kernel: int8, board_wstream/board_fparams required"
                        : "wstream/fparams must not be NULL");
    default:
        return fail(BF_ERR_ARGUMENT, "kernel must be BF_KERNEL_AUTO, BF_KERNEL_QUAD, BF_KERNEL_BOARD, BF_KERNEL_TWIN, BF_KERNEL_OCTO or BF_KERNEL_DUO");
    }
}

extern "C" int bf_kernel_choice(const bf_eval_args* args) { return choose_kernel(args); }

// Whether the encoder-only build of kernel `kind` serves this launch: nothing but the stream is tapped, and the
// kernel is one that AUTO chooses from, or TWIN in e4m3, which AUTO chose before DUO carried that format (the others run
// their taps build, whose every phase tests for taps).
static bool enc_build(const bf_eval_args* a, int kind) {
    const bf_taps* t = a->taps;
    if (!t || !t->alive || t->embed || t->qa_qkv || t->acc_qkv || t->qa_out || t->acc_out || t->qa_ff1 || t->acc_ff1 || t->qa_ff2 ||
        t->acc_ff2 || t->resid || t->normed)
        return false;
    if (a->shape.d_model == 512) return kind == BF_KERNEL_OCTO;
    return kind == BF_KERNEL_OCTO || kind == BF_KERNEL_DUO || (kind == BF_KERNEL_TWIN && a->quant == BF_QUANT_E4M3);
}

// Whether AUTO keeps this launch on one position per workgroup (256 wide: TWIN; 512 wide: OCTO) where it would pair them: too
// many layers for the kernels that do, or (e4m3 and 512 wide) flags without a list.  A workgroup of one position leaves when its flag is 0; a pair of neighbours runs when either is live.
// 4000 flags, scattered, of which 5 % / a third / two thirds / all are set: e4m3 281 / 986 / 1693 / 2174 us against 476 /
// 1616 / 1891 / 1959 of pairs, 512 wide 1.45 / 5.67 / 9.99 / 12.1 ms against 2.04 / 7.54 / 9.14 / 9.50: flags are there for
// the launches of which most is not live.  int8 of the 256-wide network: 356 / 1227 / 1503 / 1481 us in pairs, which
// AUTO has given it since it has had them; as a list 129 / 561 / 1098 / 1537.
static bool unpaired(const bf_eval_args* a) {
    return !offsets_reach(&a->shape, 1) || (a->active && (a->quant == BF_QUANT_E4M3 || a->shape.d_model == 512));
}

// What AUTO makes of choose_kernel()'s answer: TWIN's launches are the two-position kernel's (same bits; e4m3, 4096
// positions: 2142 -> 1962 us).
static int run_kernel(const bf_eval_args* a) {
    const int kind = choose_kernel(a);
    return a && a->kernel == BF_KERNEL_AUTO && kind == BF_KERNEL_TWIN && !unpaired(a) ? BF_KERNEL_DUO : kind;
}

static int check_args(const bf_eval_args* a, bf::KArgs* k, int* kind) {
    *kind = run_kernel(a);
    if (*kind < 0) return *kind;
    const bool board = *kind == BF_KERNEL_BOARD || *kind == BF_KERNEL_TWIN || *kind == BF_KERNEL_OCTO || *kind == BF_KERNEL_DUO;
    if (a->n < 1 || a->n > (1ll << 28)) return fail(BF_ERR_ARGUMENT, "n must be in [1, 2^28]");
    // encoder-only launch: residual stream in and out through the tap table, no board words, no heads
    const bool enc_only = a->taps && a->taps->alive;
    if (a->taps && (a->taps->x_in_h || a->taps->resid_last_h) && !enc_build(a, *kind))
        return fail(BF_ERR_UNSUPPORTED, "x_in_h / resid_last_h: encoder-only launches of the kernel AUTO chooses, without other taps");
    if (enc_only) {
        if (!(a->taps->x_in || a->taps->x_in_h) || !(a->taps->resid_last || a->taps->resid_last_h))
            return fail(BF_ERR_ARGUMENT, "an encoder-only launch (taps.alive) needs taps.x_in and taps.resid_last");
        if (((uintptr_t)a->taps->resid_last & 15) || (((uintptr_t)a->taps->x_in_h | (uintptr_t)a->taps->resid_last_h) & 7))
            return fail(BF_ERR_ARGUMENT, "resid_last must be 16-byte aligned, x_in_h and resid_last_h 8-byte aligned");
        if (a->leaf_index || a->leaf_count || a->active)
            return fail(BF_ERR_ARGUMENT, "an encoder-only launch takes neither active flags nor a leaf list");
    } else {
        if (!a->boards || !a->control || !a->rep) return fail(BF_ERR_ARGUMENT, "boards/control/rep must not be NULL");
        if (!a->policy || !a->promo || !a->value) return fail(BF_ERR_ARGUMENT, "policy/promo/value must not be NULL");
    }
    const uint8_t* ws = board ? a->board_wstream : a->wstream;
    const float* fp = board ? a->board_fparams : a->fparams;
    if (((uintptr_t)ws & 15) || ((uintptr_t)fp & 15))
        return fail(BF_ERR_ARGUMENT, "the parameter blobs must be 16-byte aligned");
    if (!enc_only && (((uintptr_t)a->policy & 15) || ((uintptr_t)a->promo & 7)))
        return fail(BF_ERR_ARGUMENT, "policy must be 16-byte and promo 8-byte aligned");
    if (!enc_only && (((uintptr_t)a->boards & 1) || ((uintptr_t)a->control & 1) || ((uintptr_t)a->value & 3) ||
                      ((uintptr_t)a->mask & 7) || ((uintptr_t)a->best_move & 3)))
        return fail(BF_ERR_ARGUMENT, "boards/control/value/mask/best_move must be aligned to their element size");
    if (!enc_only && a->best_move && !a->mask) return fail(BF_ERR_ARGUMENT, "best_move needs a mask");
    if ((a->leaf_index == nullptr) != (a->leaf_count == nullptr))
        return fail(BF_ERR_ARGUMENT, "leaf_index and leaf_count come together");
    if (a->leaf_index && a->active) return fail(BF_ERR_ARGUMENT, "a compacted leaf list replaces the active flags: pass one of them");
    if (((uintptr_t)a->leaf_index & 3) || ((uintptr_t)a->leaf_count & 3))
        return fail(BF_ERR_ARGUMENT, "leaf_index / leaf_count must be 4-byte aligned");
    if ((uintptr_t)a->team_workspace & 255) return fail(BF_ERR_ARGUMENT, "team_workspace must be 256-byte aligned");
    if (a->value_mode < BF_VALUE_KING || a->value_mode > BF_VALUE_PRENORM)
        return fail(BF_ERR_ARGUMENT, "value_mode must be BF_VALUE_KING, BF_VALUE_POOLED or BF_VALUE_PRENORM");
    if (a->value_mode != BF_VALUE_KING && !board)
        return fail(BF_ERR_UNSUPPORTED, "the pooled value heads run on the BOARD, TWIN, OCTO and DUO kernels");
    if (!board && (!a->workspace || ((uintptr_t)a->workspace & 15) || a->workspace_bytes < bf_workspace_bytes(&a->shape, a->n)))
        return fail(BF_ERR_ARGUMENT, "workspace must be 16-byte aligned and hold bf_workspace_bytes(shape, n) bytes");
    memset(k, 0, sizeof(*k));
    k->boards = a->boards; k->control = a->control; k->rep = a->rep; k->mask = a->mask; k->active = a->active;
    k->leaf_index = a->leaf_index; k->leaf_count = a->leaf_count;
    k->n = (int)a->n;
    k->wstream = ws; k->fparams = fp;
    k->policy = a->policy; k->promo = a->promo; k->value = a->value; k->best = a->best_move;
    k->out_fp32 = a->out_fp32 ? 1 : 0;
    k->xpark = static_cast<float*>(a->workspace);
    k->team_ws = static_cast<uint8_t*>(a->team_workspace);
    k->n_layers = a->shape.n_layers; k->n_value = a->shape.n_value; k->eps = a->shape.eps;
    k->vmode = a->value_mode;
    k->l0 = 0; k->l1 = a->shape.n_layers;
    if (a->taps) {
        k->taps = *a->taps;
        if (a->taps->layer_begin || a->taps->layer_end) {
            k->l0 = a->taps->layer_begin; k->l1 = a->taps->layer_end;
            if (k->l0 < 0 || k->l1 > k->n_layers || k->l0 > k->l1)
                return fail(BF_ERR_ARGUMENT, "taps layer range must satisfy 0 <= begin <= end <= n_layers");
        }
        if (a->taps->x_in && ((uintptr_t)a->taps->x_in & 15)) return fail(BF_ERR_ARGUMENT, "x_in must be 16-byte aligned");
    }
    if (enc_only) {   // nothing of these is read or written
        k->boards = nullptr; k->control = nullptr; k->rep = nullptr; k->mask = nullptr;
        k->policy = nullptr; k->promo = nullptr; k->value = nullptr; k->best = nullptr;
    }
    return BF_OK;
}

// Whether the current device is an MI355X-class part (gfx950), looked up once per device; the
// kernels are compiled for that architecture only.
bool bf::device_is_gfx950() {
    static std::atomic<unsigned long long> known{0}, good{0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        fail(BF_ERR_DEVICE, "no current HIP device");
        return false;
    }
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
    bool ok;
    if (known.load(std::memory_order_acquire) & bit) {
        ok = good.load(std::memory_order_relaxed) & bit;
    } else {
        hipDeviceProp_t prop;
        ok = hipGetDeviceProperties(&prop, dev) == hipSuccess && strncmp(prop.gcnArchName, "gfx950", 6) == 0;
        if (ok) good.fetch_or(bit, std::memory_order_relaxed);
        known.fetch_or(bit, std::memory_order_release);
    }
    if (!ok) fail(BF_ERR_DEVICE, "the current device is not a gfx950 GPU: the kernels of this library are built for MI355X only");
    return ok;
}

// the arguments of a launch over positions [first, first + count) of the caller's arrays
static bf::KArgs slice(const bf::KArgs& k, int d_model, int first, int count) {
    bf::KArgs s = k;
    const size_t f = (size_t)first, logit = k.out_fp32 ? 4 : 2;
    s.n = count;
    if (k.taps.alive) {   // encoder-only: the stream and the token mask are the arrays
        const size_t at = f * BF_TOKENS * d_model;
        s.taps.alive += f * BF_TOKENS;
        if (s.taps.x_in) s.taps.x_in += at;
        if (s.taps.resid_last) s.taps.resid_last += at;
        if (s.taps.x_in_h) s.taps.x_in_h = static_cast<const uint16_t*>(s.taps.x_in_h) + at;
        if (s.taps.resid_last_h) s.taps.resid_last_h = static_cast<uint16_t*>(s.taps.resid_last_h) + at;
        return s;
    }
    s.boards += f * BF_TOKENS;
    s.control += f;
    s.rep += f;
    if (s.mask) s.mask += f * BF_TOKENS;
    if (s.active) s.active += f;
    s.policy = static_cast<char*>(k.policy) + f * BF_TOKENS * BF_POLICY * logit;
    s.promo = static_cast<char*>(k.promo) + f * BF_TOKENS * BF_PROMO * logit;
    s.value += f;
    if (s.best) s.best += f;
    return s;
}

// Positions a team launch of this call may hold: 0 unless AUTO chose, a workspace came along and nothing but the
// stream is tapped.
static int team_limit(const bf_eval_args* a, bool profile, bool enc) {
    if (a->kernel != BF_KERNEL_AUTO || !a->team_workspace || profile || (a->taps && !enc) || !offsets_reach(&a->shape, 4)) return 0;
    const size_t fits = a->team_workspace_bytes / bf::team_slot_bytes(a->shape.d_model);
    const int most = bf::team_positions(a->shape.d_model, false);
    return fits < (size_t)most ? (int)fits : most;
}

// How a launch of kernel `kind` is carried out: launch() follows it and bf_launch_form() tells it.
struct Route {
    int form;       // enum bf_form
    bool enc;       // the encoder-only build
    bool rounds;    // whole rounds of two positions per workgroup (form), the rest in other workgroups behind them
    int team;       // positions a team launch may hold, 0: none
    bool by_teams(const bf_eval_args* a, int64_t n) const {   // whether n of the launch's positions go to teams
        return team > 0 && !(a->leaf_index && n > team) && n <= (a->shape.d_model == 512 ? 2 : 1) * team;
    }
};
static Route route(const bf_eval_args* a, int kind, bool profile) {
    const bool wide = a->shape.d_model == 512, pairs = a->kernel == BF_KERNEL_AUTO && a->n > kBoardMaxN && (wide ? !unpaired(a) : kind == BF_KERNEL_DUO);
    Route r;
    r.enc = !profile && enc_build(a, kind);
    r.team = team_limit(a, profile, r.enc);
    r.rounds = pairs && (!a->taps || r.enc) && !profile;
    r.form = kind;   // the forms named after a kernel have its number
    if (wide && (r.rounds || (pairs && profile))) r.form = BF_FORM_WIDE;
    else if (kind == BF_KERNEL_OCTO && !r.rounds && r.by_teams(a, a->n)) r.form = BF_FORM_TEAM;
    return r;
}

static hipError_t launch_team(const bf_eval_args* a, bf::KArgs k, bool enc, hipStream_t stream) {
    k.team_gave_up = bf::team_report_word();
    if (a->shape.d_model == 512) return (enc ? bf::launch_team512_enc : bf::launch_team512)(k, stream);
    if (a->quant == BF_QUANT_E4M3) return (enc ? bf::launch_team256_fp8_enc : bf::launch_team256_fp8)(k, stream);
    return (enc ? bf::launch_team256_enc : bf::launch_team256)(k, stream);
}

static int launch(const bf_eval_args* a, const bf::KArgs& k, int kind, hipStream_t stream) {
    const int grid = (k.n + bf::WAVES - 1) / bf::WAVES;
    hipError_t e;
    if (!bf::device_is_gfx950()) return BF_ERR_DEVICE;
    if (bf::team_gave_up())
        return fail(BF_ERR_TEAM, "an earlier launch on this device gave up waiting for compute units held by other launches and its outputs "
                                 "are NaN (see team_workspace of bf_eval_args); nothing was launched now");
    const bool wide = a->shape.d_model == 512;
    const Route to = route(a, kind, k.profile != nullptr);
    const bool enc = to.enc;
    // A launch whose teams have a compute unit for every member (64 positions, 512 wide: 32) goes to the team form (one
    // position 117 -> 74 us, 64 112 -> 79, e4m3 138 -> 89 and 140 -> 94; 512 wide, one 755 -> 260, 32 728 -> 315), and 512 wide so does one
    // that two team launches hold (33 positions 727 -> 572, 64 715 -> 620).
    auto launch_teams = [&](const bf::KArgs& s) {
        hipError_t r = hipSuccess;
        for (int at = 0; at < s.n && r == hipSuccess; at += to.team)
            r = launch_team(a, s.n <= to.team ? s : slice(s, a->shape.d_model, at, s.n - at < to.team ? s.n - at : to.team), enc, stream);
        return r;
    };
    if (to.form == BF_FORM_TEAM) {
        e = launch_teams(k);
    } else if (to.rounds) {
        // Two positions per workgroup, in rounds of 512 positions that cost the same full or not: a last round of at most 256
        // goes to the one-position form (640 positions: 0.282 ms instead of 0.335, e4m3 0.368 instead of 0.452), 256 wide in the same
        // launch (ragged_kernel).  With a leaf list the count is on the device: both forms run and each takes its share of the list (200
        // live leaves of 1000 take 114 us instead of 166).  Not with other taps or the profile.
        const int rest = k.leaf_index ? bf::DUO_ROUND / 2 : bf::round_rest(k.n);
        const bool f8 = a->quant == BF_QUANT_E4M3, teams = rest && !k.leaf_index && to.by_teams(a, rest);
        if (rest && !wide && !teams) {
            bf::KArgs both = k;
            both.list_split = k.leaf_index != nullptr;
            both.pairs = (k.leaf_index ? k.n + 1 : k.n - rest) / 2;
            both.single_from = k.leaf_index ? 0 : k.n - rest;
            both.grid = rest;
            e = (f8 ? (enc ? bf::launch_ragged256_fp8_enc : bf::launch_ragged256_fp8) : (enc ? bf::launch_ragged256_enc : bf::launch_ragged256))(both, stream);
        } else {   // of the 256-wide network: no list, and no last round but the teams'
            bf::KArgs front = k, back = k;
            if (k.leaf_index) {
                front.list_split = back.list_split = 1;
                back.grid = rest;
            } else if (rest) {
                front = slice(k, a->shape.d_model, 0, k.n - rest);
                back = slice(k, a->shape.d_model, k.n - rest, rest);
            }
            e = (wide ? (enc ? bf::launch_wide512_enc : bf::launch_wide512)
                 : f8 ? (enc ? bf::launch_duo256_fp8_enc : bf::launch_duo256_fp8)
                      : (enc ? bf::launch_duo256_enc : bf::launch_duo256))(front, stream);
            if (rest && e == hipSuccess) e = teams ? launch_teams(back) : (enc ? bf::launch_octo512_enc : bf::launch_octo512)(back, stream);
        }
    } else if (enc) {
        if (wide) e = bf::launch_octo512_enc(k, stream);
        else if (a->quant == BF_QUANT_E4M3)
            e = (kind == BF_KERNEL_OCTO ? bf::launch_solo256_fp8_enc : kind == BF_KERNEL_TWIN ? bf::launch_twin256_fp8_enc : bf::launch_duo256_fp8_enc)(k, stream);
        else e = (kind == BF_KERNEL_OCTO ? bf::launch_solo256_enc : bf::launch_duo256_enc)(k, stream);
    } else if (kind == BF_KERNEL_OCTO) {
        // eight wavefronts per position: the 512-wide network on the board kernel's eight-wavefront form; the
        // 256-wide one on the two-position kernel's one-position form, which issues each product under the
        // previous one's epilogue
        if (k.profile && wide)
            e = (to.form == BF_FORM_WIDE ? bf::launch_wide512_prof : bf::launch_octo512_prof)(k, stream);
        else if (wide)
            e = a->taps ? bf::launch_octo512_taps(k, stream) : bf::launch_octo512(k, stream);
        else if (a->quant == BF_QUANT_E4M3)
            e = k.profile ? bf::launch_solo256_fp8_prof(k, stream)
              : a->taps   ? bf::launch_solo256_fp8_taps(k, stream)
                          : bf::launch_solo256_fp8(k, stream);
        else if (k.profile)
            e = bf::launch_solo256_prof(k, stream);
        else
            e = a->taps ? bf::launch_solo256_taps(k, stream) : bf::launch_solo256(k, stream);
    } else if (kind == BF_KERNEL_DUO) {
        if (k.profile)
            e = a->quant == BF_QUANT_E4M3 ? bf::launch_duo256_fp8_prof(k, stream) : bf::launch_duo256_prof(k, stream);
        else if (a->quant == BF_QUANT_E4M3)
            e = a->taps ? bf::launch_duo256_fp8_taps(k, stream) : bf::launch_duo256_fp8(k, stream);
        else
            e = a->taps ? bf::launch_duo256_taps(k, stream) : bf::launch_duo256(k, stream);
    } else if (kind == BF_KERNEL_TWIN) {
        if (k.profile)
            e = a->quant == BF_QUANT_E4M3 ? bf::launch_twin256_fp8_prof(k, stream) : bf::launch_twin256_prof(k, stream);
        else if (a->quant == BF_QUANT_E4M3)
            e = a->taps ? bf::launch_twin256_fp8_taps(k, stream) : bf::launch_twin256_fp8(k, stream);
        else
            e = a->taps ? bf::launch_twin256_taps(k, stream) : bf::launch_twin256(k, stream);
    } else if (kind == BF_KERNEL_BOARD) {
        if (k.profile)
            e = a->shape.d_model == 512      ? bf::launch_board512_prof(k, stream)
              : a->quant == BF_QUANT_E4M3 ? bf::launch_board256_fp8_prof(k, stream)
                                          : bf::launch_board256_prof(k, stream);
        else if (a->shape.d_model == 512)
            e = a->taps ? bf::launch_board512_taps(k, stream) : bf::launch_board512(k, stream);
        else if (a->quant == BF_QUANT_E4M3)
            e = a->taps ? bf::launch_board256_fp8_taps(k, stream) : bf::launch_board256_fp8(k, stream);
        else
            e = a->taps ? bf::launch_board256_taps(k, stream) : bf::launch_board256(k, stream);
    } else if (a->quant == BF_QUANT_E4M3)
        e = k.profile ? bf::launch_prof_fp8(k, grid, stream)
          : a->taps   ? bf::launch_taps_fp8(k, grid, stream)
                      : bf::launch_prod_fp8(k, grid, stream);
    else
        e = k.profile ? bf::launch_prof(k, grid, stream)
          : a->taps   ? bf::launch_taps(k, grid, stream)
                      : bf::launch_prod(k, grid, stream);
    if (e != hipSuccess) {
        snprintf(g_err, sizeof(g_err), "kernel launch failed: %s", hipGetErrorString(e));
        return BF_ERR_LAUNCH;
    }
    return BF_OK;
}

extern "C" int bf_launch_form(const bf_eval_args* args) {
    const int kind = run_kernel(args);
    return kind < 0 ? kind : route(args, kind, false).form;
}

extern "C" int bf_model_forward(const bf_eval_args* args, void* stream) {
    bf::KArgs k;
    int kind;
    const int rc = check_args(args, &k, &kind);
    if (rc) return rc;
    return launch(args, k, kind, (hipStream_t)stream);
}

// ---- the entry point that allocates nothing ----------------------------------------------------
// The four-positions-per-workgroup kernel parks the residual stream in a workspace the caller
// lends to bf_model_forward.  For callers that cannot allocate, the same launch with the
// workspace in this file-scope device array.  Each GPU the library runs on holds its own copy
// at its own address until the process ends; `scratch` is the host-side stand-in of the symbol
// and is never passed to a kernel: host code uses the per-device address looked up below.
static __device__ __align__(256) uint8_t scratch[(size_t)BF_STATIC_MAX_N * bf::T * bf::D * sizeof(float)];

static const int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices];   // device address of `scratch` on device i, NULL until looked up

// The address of this device's copy of `scratch`, looked up once per device with that device
// current (the caller's current device is the one the launch goes to).
static int scratch_address(void** out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(BF_ERR_DEVICE, "no current HIP device (or its ordinal is 64 or more)");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            snprintf(g_err, sizeof(g_err), "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
            return BF_ERR_LAUNCH;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return BF_OK;
}

extern "C" int bf_model_forward_static(const bf_eval_args* args, void* stream) {
    if (!args) return fail(BF_ERR_ARGUMENT, "args is NULL");
    if (args->kernel != BF_KERNEL_AUTO && args->kernel != BF_KERNEL_QUAD)
        return fail(BF_ERR_ARGUMENT, "bf_model_forward_static runs the four-positions-per-workgroup kernel: kernel must be BF_KERNEL_QUAD "
                                     "or BF_KERNEL_AUTO (the other kernels need no workspace: call bf_model_forward)");
    if (args->n > BF_STATIC_MAX_N) {
        snprintf(g_err, sizeof(g_err), "n = %lld exceeds BF_STATIC_MAX_N = %d positions, the size of the library's static workspace",
                 (long long)args->n, BF_STATIC_MAX_N);
        return BF_ERR_ARGUMENT;
    }
    // the argument checks come first (they touch no device); the placeholder only has to pass them
    bf_eval_args a = *args;
    a.kernel = BF_KERNEL_QUAD;
    a.workspace = reinterpret_cast<void*>(uintptr_t(256));
    a.workspace_bytes = sizeof(scratch);
    bf::KArgs k;
    int kind;
    const int rc = check_args(&a, &k, &kind);
    if (rc) return rc;
    void* ws = nullptr;
    const int rc0 = scratch_address(&ws);
    if (rc0) return rc0;
    k.xpark = static_cast<float*>(ws);
    return launch(&a, k, kind, (hipStream_t)stream);
}

extern "C" int bf_profile_phases(const bf_eval_args* args, void* stream, uint64_t* cycles) {
    bf::KArgs k;
    int kind;
    const int rc = check_args(args, &k, &kind);
    if (rc) return rc;
    if (args->taps) return fail(BF_ERR_ARGUMENT, "the phase profile runs without taps");
    if (!cycles) return fail(BF_ERR_ARGUMENT, "cycles must not be NULL");
    k.profile = reinterpret_cast<unsigned long long*>(cycles);
    return launch(args, k, kind, (hipStream_t)stream);
}

extern "C" int bf_profile_phase_count(void) { return bf::N_PHASES; }

extern "C" const char* bf_profile_phase_name(int i) {
    static const char* names[bf::N_PHASES] = {"embed", "ln1_quant", "qkv_gemm_epilogue", "attention",
                                              "oquant_outproj", "ln2_quant", "ffn1", "ffn2", "heads",
                                              "store", "sync_wait", "total"};
    return (i >= 0 && i < bf::N_PHASES) ? names[i] : "";
}

extern "C" double bf_time_kernel_ms(const bf_eval_args* args, void* stream, int warmup, int iters) {
    bf::KArgs k;
    int kind;
    int rc = check_args(args, &k, &kind);
    if (rc) return rc;
    if (iters < 1 || warmup < 0) return fail(BF_ERR_ARGUMENT, "iters must be >= 1 and warmup >= 0");
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return fail(BF_ERR_LAUNCH, "hipEventCreate failed");
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail(BF_ERR_LAUNCH, "hipEventCreate failed");
    }
    for (int i = 0; i < warmup && !rc; i++) rc = launch(args, k, kind, s);
    (void)hipEventRecord(e0, s);
    for (int i = 0; i < iters && !rc; i++) rc = launch(args, k, kind, s);
    (void)hipEventRecord(e1, s);
    const hipError_t e = hipEventSynchronize(e1);
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    if (e != hipSuccess) return fail(BF_ERR_LAUNCH, hipGetErrorString(e));
    return (double)ms / iters;
}
