// PyTorch (ROCm) extension module over the C-ABI of include/brokefish_hip.h: the counterpart of the
// reference's pybind module (reference csrc/encoder.cu:1770-1876 model_forward, :1905-1930 the
// exported functions; loaded by brokefish/nn/_build.py:149-190).  Tensors in, one asynchronous
// launch on the current HIP stream of the tensors' device, caller-allocated outputs, argument
// errors as TORCH_CHECK failures (Python RuntimeError).  No device code here: the kernels live in
// libbrokefish_hip.so, which this module links.
#include <torch/extension.h>

// PyTorch on ROCm presents its devices under the type name "cuda": these are the guard and stream
// classes of that arrangement
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <pybind11/stl.h>

#include <algorithm>
#include <array>
#include <optional>
#include <string>
#include <string_view>
#include <utility>
#include <vector>

#include "brokefish_hip.h"

namespace {

typedef c10::optional<torch::Tensor> OptTensor;

// None (or an empty tensor, as in the reference binding, csrc/encoder.cu:1607-1612) means "absent".
torch::Tensor get(const OptTensor& t) { return t.has_value() ? *t : torch::Tensor(); }
bool absent(const torch::Tensor& t) { return !t.defined() || t.numel() == 0; }
const void* ptr_or_null(const torch::Tensor& t) { return absent(t) ? nullptr : t.data_ptr(); }

struct Checked {
    bf_eval_args a;
    c10::Device device;
};

Checked check(const torch::Tensor& boards, const torch::Tensor& control, const torch::Tensor& rep,
              const torch::Tensor& weights, const torch::Tensor& params, const torch::Tensor& policy,
              const torch::Tensor& promo, const torch::Tensor& value, int64_t d_model, int64_t n_layers,
              int64_t n_heads, int64_t d_ff, double eps, int64_t quant, int64_t kernel, int64_t n_value,
              int64_t vmode, const OptTensor& mask_, const OptTensor& best_move_, const OptTensor& active_,
              const OptTensor& workspace_, const OptTensor& leaf_index_ = c10::nullopt,
              const OptTensor& leaf_count_ = c10::nullopt, const OptTensor& team_workspace_ = c10::nullopt) {
    const torch::Tensor mask = get(mask_), best_move = get(best_move_), active = get(active_), workspace = get(workspace_);
    const torch::Tensor leaf_index = get(leaf_index_), leaf_count = get(leaf_count_);
    TORCH_CHECK(boards.is_cuda() && boards.scalar_type() == torch::kShort && boards.is_contiguous() &&
                    boards.dim() == 2 && boards.size(1) == BF_TOKENS,
                "boards must be [n, 32] int16 contiguous on the GPU");
    const int64_t n = boards.size(0);
    TORCH_CHECK(n >= 1, "boards must hold at least one position");
    const auto dev = boards.device();
    auto on_dev = [&](const torch::Tensor& t) { return t.is_cuda() && t.device() == dev && t.is_contiguous(); };
    TORCH_CHECK(on_dev(control) && control.scalar_type() == torch::kShort && control.numel() == n,
                "control must be [n] int16 contiguous on the boards' device");
    TORCH_CHECK(on_dev(rep) && rep.scalar_type() == torch::kByte && rep.numel() == n,
                "rep must be [n] uint8 contiguous on the boards' device");
    TORCH_CHECK(on_dev(weights) && weights.scalar_type() == torch::kByte, "weights must be a uint8 blob on the boards' device");
    TORCH_CHECK(on_dev(params) && params.scalar_type() == torch::kFloat, "params must be a float32 blob on the boards' device");
    TORCH_CHECK(on_dev(policy) && on_dev(promo) && policy.scalar_type() == promo.scalar_type() &&
                    (policy.scalar_type() == torch::kHalf || policy.scalar_type() == torch::kFloat) &&
                    policy.numel() == n * BF_TOKENS * BF_POLICY && promo.numel() == n * BF_TOKENS * BF_PROMO,
                "policy must be [n, 32, 64] and promo [n, 32, 4], both fp16 or both fp32, contiguous");
    TORCH_CHECK(on_dev(value) && value.scalar_type() == torch::kFloat && value.numel() == n, "value must be [n] float32");
    if (!absent(mask))
        TORCH_CHECK(on_dev(mask) && mask.scalar_type() == torch::kLong && mask.numel() == n * BF_TOKENS,
                    "mask must be [n, 32] int64 (legal-move words)");
    if (!absent(best_move))
        TORCH_CHECK(!absent(mask) && on_dev(best_move) && best_move.scalar_type() == torch::kInt && best_move.numel() == n,
                    "best_move must be [n] int32 and needs a mask");
    if (!absent(active))
        TORCH_CHECK(on_dev(active) && (active.scalar_type() == torch::kByte || active.scalar_type() == torch::kBool) &&
                        active.numel() == n,
                    "active must be [n] uint8 or bool");
    if (!absent(workspace)) TORCH_CHECK(on_dev(workspace) && workspace.scalar_type() == torch::kByte, "workspace must be uint8");
    TORCH_CHECK(absent(leaf_index) == absent(leaf_count), "leaf_index and leaf_count come together");
    if (!absent(leaf_index))
        TORCH_CHECK(on_dev(leaf_index) && on_dev(leaf_count) && leaf_index.scalar_type() == torch::kInt &&
                        leaf_count.scalar_type() == torch::kInt && leaf_index.numel() >= n && leaf_count.numel() == 1,
                    "leaf_index must be [n] int32 and leaf_count [1] int32 (see bf_compact_leaves)");

    Checked c{bf_eval_args{}, dev};
    bf_eval_args& a = c.a;
    a.boards = static_cast<const uint16_t*>(boards.data_ptr());
    a.control = static_cast<const int16_t*>(control.data_ptr());
    a.rep = static_cast<const uint8_t*>(rep.data_ptr());
    a.mask = static_cast<const uint64_t*>(ptr_or_null(mask));
    a.n = n;
    a.shape = bf_shape{(int32_t)d_model, (int32_t)n_layers, (int32_t)n_heads, (int32_t)d_ff, (int32_t)n_value, (float)eps};
    // one pair of blobs, in the layout of the kernel that is to run
    if (kernel == BF_KERNEL_QUAD) {
        a.wstream = static_cast<const uint8_t*>(weights.data_ptr());
        a.fparams = static_cast<const float*>(params.data_ptr());
        TORCH_CHECK((size_t)weights.numel() == bf_wstream_bytes(&a.shape) && (size_t)params.numel() == bf_fparams_floats(&a.shape),
                    "weights / params are not the blobs of this shape for the four-positions-per-workgroup kernel");
        TORCH_CHECK(!absent(workspace) && (size_t)workspace.numel() >= bf_workspace_bytes(&a.shape, n),
                    "the four-positions-per-workgroup kernel needs a workspace of bf_workspace_bytes(shape, n) bytes");
        a.workspace = workspace.data_ptr();
        a.workspace_bytes = (size_t)workspace.numel();
    } else {
        a.board_wstream = static_cast<const uint8_t*>(weights.data_ptr());
        a.board_fparams = static_cast<const float*>(params.data_ptr());
        TORCH_CHECK((size_t)weights.numel() == bf_board_wstream_bytes(&a.shape) &&
                        (size_t)params.numel() == bf_board_fparams_floats(&a.shape),
                    "weights / params are not the blobs of this shape for the one-position-per-workgroup kernels");
    }
    a.policy = policy.data_ptr();
    a.promo = promo.data_ptr();
    a.value = static_cast<float*>(value.data_ptr());
    a.best_move = absent(best_move) ? nullptr : static_cast<int32_t*>(best_move.data_ptr());
    a.out_fp32 = policy.scalar_type() == torch::kFloat;
    a.quant = (int32_t)quant;
    a.active = static_cast<const uint8_t*>(ptr_or_null(active));
    a.kernel = (int32_t)kernel;
    a.value_mode = (int32_t)vmode;
    a.leaf_index = static_cast<const int32_t*>(ptr_or_null(leaf_index));
    a.leaf_count = static_cast<const int32_t*>(ptr_or_null(leaf_count));
    const torch::Tensor team = get(team_workspace_);
    if (!absent(team)) {
        TORCH_CHECK(on_dev(team) && team.scalar_type() == torch::kByte, "team_workspace must be uint8 on the boards' device");
        a.team_workspace = team.data_ptr();
        a.team_workspace_bytes = (size_t)team.numel();
    }
    return c;
}

void model_forward(torch::Tensor boards, torch::Tensor control, torch::Tensor rep, torch::Tensor weights,
                   torch::Tensor params, torch::Tensor policy, torch::Tensor promo, torch::Tensor value,
                   int64_t d_model, int64_t n_layers, int64_t n_heads, int64_t d_ff, double eps, int64_t quant,
                   int64_t kernel, int64_t n_value, int64_t vmode, OptTensor mask, OptTensor best_move,
                   OptTensor active, OptTensor workspace, OptTensor leaf_index, OptTensor leaf_count, OptTensor team_workspace) {
    const Checked c = check(boards, control, rep, weights, params, policy, promo, value, d_model, n_layers, n_heads,
                            d_ff, eps, quant, kernel, n_value, vmode, mask, best_move, active, workspace, leaf_index, leaf_count, team_workspace);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(c.device);     // the launch goes to the tensors' device
    const int rc = bf_model_forward(&c.a, c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(c.device.index()).stream());
    TORCH_CHECK(rc == BF_OK, "bf_model_forward failed (", rc, "): ", bf_last_error());
}

// The encoder stack alone, in place on y (reference csrc/encoder.cu:1752-1764 encoder_forward(y,
// weights, alive, n_layers, eps, debug_stage)): y [n, 32, d_model] float32 is the residual stream
// entering the first layer and, on return, the stream leaving the last; alive [n, 32] int8 or bool
// masks dead tokens out of attention as keys.  No heads run and nothing is allocated.
void encoder_forward(torch::Tensor y, torch::Tensor weights, torch::Tensor params, torch::Tensor alive,
                     int64_t d_model, int64_t n_layers, int64_t n_heads, int64_t d_ff, double eps, int64_t quant,
                     int64_t kernel, int64_t n_value, OptTensor workspace_) {
    const torch::Tensor workspace = get(workspace_);
    TORCH_CHECK(y.is_cuda() && y.scalar_type() == torch::kFloat && y.is_contiguous() && y.dim() == 3 &&
                    y.size(1) == BF_TOKENS && y.size(2) == d_model && y.size(0) >= 1,
                "y must be [n, 32, d_model] float32 contiguous on the GPU");
    const auto dev = y.device();
    auto on_dev = [&](const torch::Tensor& t) { return t.is_cuda() && t.device() == dev && t.is_contiguous(); };
    TORCH_CHECK(on_dev(alive) && (alive.scalar_type() == torch::kChar || alive.scalar_type() == torch::kBool) &&
                    alive.numel() == y.size(0) * BF_TOKENS,
                "alive must be [n, 32] int8 or bool on y's device");
    TORCH_CHECK(on_dev(weights) && weights.scalar_type() == torch::kByte, "weights must be a uint8 blob on y's device");
    TORCH_CHECK(on_dev(params) && params.scalar_type() == torch::kFloat, "params must be a float32 blob on y's device");
    bf_eval_args a{};
    bf_taps taps{};
    a.n = y.size(0);
    a.shape = bf_shape{(int32_t)d_model, (int32_t)n_layers, (int32_t)n_heads, (int32_t)d_ff, (int32_t)n_value, (float)eps};
    if (kernel == BF_KERNEL_QUAD) {
        a.wstream = static_cast<const uint8_t*>(weights.data_ptr());
        a.fparams = static_cast<const float*>(params.data_ptr());
        TORCH_CHECK((size_t)weights.numel() == bf_wstream_bytes(&a.shape) && (size_t)params.numel() == bf_fparams_floats(&a.shape),
                    "weights / params are not the blobs of this shape for the four-positions-per-workgroup kernel");
        TORCH_CHECK(!absent(workspace) && on_dev(workspace) && (size_t)workspace.numel() >= bf_workspace_bytes(&a.shape, a.n),
                    "the four-positions-per-workgroup kernel needs a workspace of bf_workspace_bytes(shape, n) bytes");
        a.workspace = workspace.data_ptr();
        a.workspace_bytes = (size_t)workspace.numel();
    } else {
        a.board_wstream = static_cast<const uint8_t*>(weights.data_ptr());
        a.board_fparams = static_cast<const float*>(params.data_ptr());
        TORCH_CHECK((size_t)weights.numel() == bf_board_wstream_bytes(&a.shape) &&
                        (size_t)params.numel() == bf_board_fparams_floats(&a.shape),
                    "weights / params are not the blobs of this shape for the one-position-per-workgroup kernels");
    }
    a.quant = (int32_t)quant;
    a.kernel = (int32_t)kernel;
    taps.x_in = static_cast<const float*>(y.data_ptr());
    taps.resid_last = static_cast<float*>(y.data_ptr());
    taps.alive = static_cast<const int8_t*>(alive.data_ptr());
    a.taps = &taps;   // copied by the library before the call returns
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dev);
    const int rc = bf_model_forward(&a, c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream());
    TORCH_CHECK(rc == BF_OK, "bf_model_forward failed (", rc, "): ", bf_last_error());
}

// ---- the calls either side of the evaluator ----------------------------------------------------------
// These launches take 5 to 10 us on the device, so at a search's sizes the host's share decides: checks,
// allocation and launch in one native call (about 4 us; through ctypes, with the guard and the stream
// looked up in Python, 10 us for movegen and 36 us for expand_edges, six zero-filling launches of
// which the kernel then overwrote).

#define BF_VALUE_CHECK(cond, ...) \
    do {                          \
        if (!(cond)) throw py::value_error(c10::str(__VA_ARGS__)); \
    } while (0)

bool shape_is(const torch::Tensor& t, std::initializer_list<int64_t> want) { return t.sizes() == at::IntArrayRef(want); }

void* stream_of(const c10::Device& dev) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream(); }

// a new tensor straight from the caching allocator, on the current device (at::empty takes the dispatcher's way there)
torch::Tensor fresh(at::IntArrayRef size, at::ScalarType type) {
    static c10::Allocator* const allocator = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
    const size_t bytes = c10::multiply_integers(size) * c10::elementSize(type);
    torch::Tensor t = at::detail::make_tensor<c10::TensorImpl>(
        c10::Storage(c10::make_intrusive<c10::StorageImpl>(c10::StorageImpl::use_byte_size_t(), bytes, allocator->allocate(bytes), allocator, true)),
        c10::DispatchKeySet(c10::DispatchKey::CUDA), c10::scalarTypeToTypeMeta(type));
    t.unsafeGetTensorImpl()->set_sizes_contiguous(size);
    return t;
}

// New tensors that a call returns together, each in memory of its own: a caller may keep, save, resize or share one
// of them and let the others go.  (Views of one allocation are 1 us cheaper for the six of an expansion, of a
// call's 6; but then keeping the edge counts keeps a hundred times their size.)  Zeroed ones are cleared by one launch.
struct Want { at::DimVector size; at::ScalarType type; };
template <size_t N>
std::array<torch::Tensor, N> fresh_together(const std::array<Want, N>& want, bool zeroed, const c10::Device& dev) {
    std::array<torch::Tensor, N> t;
    for (size_t i = 0; i < N; i++) t[i] = fresh(want[i].size, want[i].type);
    if (zeroed) {
        void* at[N];
        size_t bytes[N];
        for (size_t i = 0; i < N; i++) {
            at[i] = t[i].data_ptr();
            bytes[i] = t[i].nbytes();
        }
        const int rc = bf_clear(at, bytes, N, stream_of(dev));
        TORCH_CHECK(rc == BF_OK, "bf_clear failed (", rc, "): ", bf_last_error());
    }
    return t;
}

void check_boards(const torch::Tensor& boards, const torch::Tensor& control, int64_t n) {
    BF_VALUE_CHECK(shape_is(boards, {n, BF_TOKENS}) && boards.scalar_type() == torch::kShort && shape_is(control, {n}) &&
                       control.scalar_type() == torch::kShort, "boards must be [n,32] int16 and control [n] int16");
    BF_VALUE_CHECK(boards.is_cuda() && control.is_cuda(), "boards and control must be on the GPU");
    BF_VALUE_CHECK(boards.is_contiguous() && control.is_contiguous(), "boards and control must be contiguous");
}
// legal-move words and check flags
std::array<torch::Tensor, 2> fresh_moves(int64_t n, const c10::Device& dev) {
    return fresh_together<2>({{{{n, BF_TOKENS}, torch::kLong}, {{n}, torch::kBool}}}, false, dev);
}

// hip_impl.movegen: (mask [n, 32] int64, in_check [n] bool)
std::pair<torch::Tensor, torch::Tensor> movegen(const torch::Tensor& boards, const torch::Tensor& control,
                                                const c10::optional<std::pair<torch::Tensor, torch::Tensor>>& out) {
    const int64_t n = boards.dim() ? boards.size(0) : 0;
    check_boards(boards, control, n);
    const c10::Device dev = boards.device();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dev);
    torch::Tensor mask, chk;
    if (out) std::tie(mask, chk) = *out;
    else {
        auto made = fresh_moves(n, dev);
        mask = std::move(made[0]);
        chk = std::move(made[1]);
    }
    BF_VALUE_CHECK(shape_is(mask, {n, BF_TOKENS}) && mask.scalar_type() == torch::kLong && shape_is(chk, {n}) && chk.scalar_type() == torch::kBool,
                   "`out` was made for another n");
    const int rc = bf_movegen(static_cast<const uint16_t*>(boards.data_ptr()), static_cast<const int16_t*>(control.data_ptr()), n,
                              static_cast<uint64_t*>(mask.data_ptr()), static_cast<uint8_t*>(chk.data_ptr()), stream_of(dev));
    TORCH_CHECK(rc == BF_OK, "bf_movegen failed (", rc, "): ", bf_last_error());
    return {mask, chk};
}

typedef c10::optional<std::pair<torch::Tensor, torch::Tensor>> OptLeaves;

void check_leaves(const torch::Tensor& index, const torch::Tensor& count, int64_t n, const c10::Device& dev) {
    BF_VALUE_CHECK(index.scalar_type() == torch::kInt && count.scalar_type() == torch::kInt && index.dim() == 1 && index.size(0) >= n &&
                       count.numel() == 1 && index.device() == dev && count.device() == dev && index.is_contiguous(),
                   "leaves must be (index [", n, "] int32, count [1] int32) on ", dev.str());
}

// hip_impl.compact_leaves: (leaf_index [n] int32, leaf_count [1] int32)
std::pair<torch::Tensor, torch::Tensor> compact_leaves(const torch::Tensor& flags_, const OptLeaves& out) {
    BF_VALUE_CHECK(flags_.dim() == 1 && (flags_.scalar_type() == torch::kByte || flags_.scalar_type() == torch::kBool) && flags_.is_cuda(),
                   "flags must be [n] uint8 or bool on the GPU");
    const int64_t n = flags_.size(0);
    const torch::Tensor flags = flags_.contiguous();
    const c10::Device dev = flags.device();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dev);
    const auto opts = flags.options().dtype(torch::kInt);
    const torch::Tensor index = out ? out->first : at::zeros({n}, opts), count = out ? out->second : at::zeros({1}, opts);
    check_leaves(index, count, n, dev);
    const int rc = bf_compact_leaves(static_cast<const uint8_t*>(flags.data_ptr()), n, static_cast<int32_t*>(index.data_ptr()),
                                     static_cast<int32_t*>(count.data_ptr()), stream_of(dev));
    TORCH_CHECK(rc == BF_OK, "bf_compact_leaves failed (", rc, "): ", bf_last_error());
    return {index, count};
}

// hip_impl.expand_edges: the dict of edge tensors.  GENERATE: mask_ and in_check are generated first, in the same launch
template <bool GENERATE = false>
py::dict expand_edges(const torch::Tensor& policy_, const torch::Tensor& promo_, const torch::Tensor& value_, const torch::Tensor& mask_,
                      const torch::Tensor& boards_, const torch::Tensor& control_, int64_t max_edges, const OptTensor& active_,
                      const c10::optional<py::dict>& out, const OptLeaves& leaves, const torch::Tensor* in_check = nullptr) {
    const int64_t n = policy_.dim() ? policy_.size(0) : 0;
    const auto lt = policy_.scalar_type();
    BF_VALUE_CHECK(shape_is(policy_, {n, BF_TOKENS, BF_POLICY}) && shape_is(promo_, {n, BF_TOKENS, BF_PROMO}) && lt == promo_.scalar_type() &&
                       (lt == torch::kHalf || lt == torch::kFloat), "policy must be [n,32,64] and promo [n,32,4], both fp16 or both fp32");
    BF_VALUE_CHECK(shape_is(value_, {n}) && value_.scalar_type() == torch::kFloat, "value must be [", n, "] float32");
    BF_VALUE_CHECK(shape_is(mask_, {n, BF_TOKENS}) && mask_.scalar_type() == torch::kLong && shape_is(boards_, {n, BF_TOKENS}) &&
                       boards_.scalar_type() == torch::kShort && shape_is(control_, {n}) && control_.scalar_type() == torch::kShort,
                   "mask must be [n,32] int64, boards [n,32] int16, control [n] int16");
    BF_VALUE_CHECK(max_edges >= 1 && max_edges <= 255, "max_edges must be in [1, 255] (edge indices are uint8 in the search)");
    BF_VALUE_CHECK(policy_.is_cuda() && promo_.is_cuda() && value_.is_cuda() && mask_.is_cuda() && boards_.is_cuda() && control_.is_cuda() &&
                       (!active_ || active_->is_cuda()), "all inputs must be on the GPU");
    const c10::Device dev = policy_.device();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dev);
    static const std::array<PyObject*, 6> keys = {PyUnicode_InternFromString("edge_move"), PyUnicode_InternFromString("edge_prior"),
                                                  PyUnicode_InternFromString("n_edges"), PyUnicode_InternFromString("count"),
                                                  PyUnicode_InternFromString("dropped"), PyUnicode_InternFromString("node_value")};
    std::array<torch::Tensor, 6> made;
    py::dict res;
    if (out) {
        res = *out;
        for (size_t i = 0; i < 6; i++) made[i] = py::cast<torch::Tensor>(res[py::handle(keys[i])]);
        BF_VALUE_CHECK(shape_is(made[0], {n, max_edges}), "`out` was made for another n or max_edges");
    } else {
        // every row is written unless positions are skipped: only then do the buffers start at zero
        made = fresh_together<6>({{{{n, max_edges}, torch::kShort}, {{n, max_edges}, torch::kHalf}, {{n}, torch::kInt}, {{n}, torch::kInt},
                                   {{n}, torch::kFloat}, {{n}, torch::kHalf}}}, active_.has_value() || leaves.has_value(), dev);
        for (size_t i = 0; i < 6; i++) {
            const py::object t = py::reinterpret_steal<py::object>(THPVariable_Wrap(made[i]));
            if (!t || PyDict_SetItem(res.ptr(), keys[i], t.ptr())) throw py::error_already_set();
        }
    }
    // temporaries made here were allocated on the current stream, where the launch is queued: their memory
    // is handed out again only to work that this stream runs after the kernel
    const c10::MaybeOwned<torch::Tensor> policy = policy_.expect_contiguous(), promo = promo_.expect_contiguous(), value = value_.expect_contiguous(),
                                         mask = mask_.expect_contiguous(), boards = boards_.expect_contiguous(), control = control_.expect_contiguous();
    bf_expand_args a{};
    a.policy = policy->data_ptr();
    a.promo = promo->data_ptr();
    a.value = static_cast<const float*>(value->data_ptr());
    a.mask = static_cast<const uint64_t*>(mask->data_ptr());
    a.boards = static_cast<const uint16_t*>(boards->data_ptr());
    a.control = static_cast<const int16_t*>(control->data_ptr());
    torch::Tensor act;
    if (active_) {
        act = active_->scalar_type() == torch::kBool ? active_->contiguous() : active_->to(torch::kByte).contiguous();
        BF_VALUE_CHECK(shape_is(act, {n}), "active must be [", n, "]");
        a.active = static_cast<const uint8_t*>(act.data_ptr());
    }
    if (leaves) {
        BF_VALUE_CHECK(!active_, "a compacted leaf list replaces the active flags: pass one of them");
        check_leaves(leaves->first, leaves->second, n, dev);
        a.leaf_index = static_cast<const int32_t*>(leaves->first.data_ptr());
        a.leaf_count = static_cast<const int32_t*>(leaves->second.data_ptr());
    }
    a.n = n;
    a.max_edges = (int32_t)max_edges;
    a.logits_fp32 = lt == torch::kFloat;
    a.edge_move = static_cast<int16_t*>(made[0].data_ptr());
    a.edge_prior = made[1].data_ptr();
    a.n_edges = static_cast<int32_t*>(made[2].data_ptr());
    a.count = static_cast<int32_t*>(made[3].data_ptr());
    a.dropped = static_cast<float*>(made[4].data_ptr());
    a.node_value = made[5].data_ptr();
    int rc;
    if constexpr (GENERATE) {
        a.mask = nullptr;
        rc = bf_movegen_expand(&a, static_cast<uint64_t*>(mask->data_ptr()), static_cast<uint8_t*>(in_check->data_ptr()), stream_of(dev));
    } else {
        rc = bf_expand(&a, stream_of(dev));
    }
    TORCH_CHECK(rc == BF_OK, "bf_expand failed (", rc, "): ", bf_last_error());
    return res;
}

// movegen and expand_edges in one launch: the dict of edge tensors with mask and in_check
py::dict movegen_expand(const torch::Tensor& policy, const torch::Tensor& promo, const torch::Tensor& value, const torch::Tensor& boards,
                        const torch::Tensor& control, int64_t max_edges, const c10::optional<py::dict>& out) {
    const int64_t n = policy.dim() ? policy.size(0) : 0;
    check_boards(boards, control, n);
    BF_VALUE_CHECK(policy.is_cuda() && policy.device() == boards.device() && control.device() == boards.device(), "all inputs must be on one GPU");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(boards.device());
    const auto made = fresh_moves(n, boards.device());
    py::dict res = expand_edges<true>(policy, promo, value, made[0], boards, control, max_edges, c10::nullopt, out, c10::nullopt, &made[1]);
    // a caller's subclass of dict may keep more than the dict (an OrderedDict its order): its own update() sees the two
    const bool plain = PyDict_CheckExact(res.ptr());
    const py::dict moves = plain ? res : py::dict();
    for (const auto& kv : {std::make_pair("mask", &made[0]), std::make_pair("in_check", &made[1])}) {
        const py::object t = py::reinterpret_steal<py::object>(THPVariable_Wrap(*kv.second));
        if (!t || PyDict_SetItemString(moves.ptr(), kv.first, t.ptr())) throw py::error_already_set();
    }
    if (!plain) res.attr("update")(moves);
    return res;
}

// ---- packing and the fingerprint ---------------------------------------------------------------------
// `params` are the network's parameters in the order of bf_layer_weights, layer by layer, and of
// bf_global_weights; those that are not fp32, contiguous, aligned and on `device` are copied there first.
// The blobs are complete when this returns, so that any stream may use them.
std::pair<torch::Tensor, torch::Tensor> pack_board(const std::vector<torch::Tensor>& params, int64_t d_model, int64_t n_layers,
                                                   int64_t d_ff, int64_t n_value, double eps, bool fp8, int64_t device) {
    const bf_shape shape{(int32_t)d_model, (int32_t)n_layers, (int32_t)(d_model / 32), (int32_t)d_ff, (int32_t)n_value, (float)eps};
    const int64_t d = d_model, f = d_ff, nl = 12 * n_layers;
    BF_VALUE_CHECK((int64_t)params.size() == nl + 10, "pack_board takes ", nl + 10, " parameters, got ", params.size());
    const int64_t layer[12][2] = {{d, 0}, {d, 0}, {3 * d, d}, {3 * d, 0}, {d, d}, {d, 0}, {d, 0}, {d, 0}, {f, d}, {f, 0}, {d, f}, {d, 0}};
    const int64_t global[10][2] = {{64, d}, {12, d}, {4, d}, {101, d}, {3, d}, {d, 0}, {d, 0}, {BF_POLICY, d}, {BF_PROMO, d}, {n_value, d}};
    const c10::Device dev(c10::kCUDA, (c10::DeviceIndex)device);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dev);
    at::NoGradGuard no_grad;
    std::vector<torch::Tensor> keep;
    std::vector<const float*> ptrs;
    ptrs.reserve(params.size());
    for (size_t i = 0; i < params.size(); i++) {
        const int64_t* want = (int64_t)i < nl ? layer[i % 12] : global[i - nl];
        torch::Tensor t = params[i];
        BF_VALUE_CHECK(want[1] ? shape_is(t, {want[0], want[1]}) : shape_is(t, {want[0]}), "a parameter is ", t.sizes(),
                       ", the network shape wants ", want[0], want[1] ? " rows of " : " elements", want[1] ? std::to_string(want[1]) : "");
        if (t.scalar_type() != torch::kFloat || t.device() != dev || !t.is_contiguous() || ((uintptr_t)t.data_ptr() & 15)) {
            t = t.detach().to(at::TensorOptions().device(dev).dtype(torch::kFloat)).contiguous();
            if ((uintptr_t)t.data_ptr() & 15) t = t.clone();
            keep.push_back(t);
        }
        ptrs.push_back(static_cast<const float*>(t.data_ptr()));
    }
    const auto opts = at::TensorOptions().device(dev);
    const torch::Tensor ws = at::empty({(int64_t)bf_board_wstream_bytes(&shape)}, opts.dtype(torch::kByte)),
                        fp = at::empty({(int64_t)bf_board_fparams_floats(&shape)}, opts.dtype(torch::kFloat)),
                        scratch = at::empty({(int64_t)bf_pack_scratch_floats(&shape)}, opts.dtype(torch::kFloat));
    const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index());
    const int rc = bf_pack_board(&shape, fp8 ? BF_QUANT_E4M3 : BF_QUANT_INT8, reinterpret_cast<const bf_layer_weights*>(ptrs.data()),
                                 reinterpret_cast<const bf_global_weights*>(ptrs.data() + nl), static_cast<uint8_t*>(ws.data_ptr()),
                                 static_cast<float*>(fp.data_ptr()), static_cast<float*>(scratch.data_ptr()), stream.stream());
    TORCH_CHECK(rc == BF_OK, "bf_pack_board failed (", rc, "): ", bf_last_error());
    {
        py::gil_scoped_release no_gil;
        stream.synchronize();
    }
    return {ws, fp};
}

// A module's parameters by name, as torch.nn.Module.named_parameters has them (modules in pre-order, each once; with `once`
// each parameter once), without its generators: some 8 us for 107 parameters where they take 57.  Where a module's type
// walks in a way of its own there is no list.
class Named {
    struct Seen {   // objects met: open addressing, grown at half full
        std::vector<PyObject*> table = std::vector<PyObject*>(512);
        size_t count = 0;
        bool insert(PyObject* p) {
            if (2 * ++count > table.size()) {
                std::vector<PyObject*> old(2 * table.size());
                old.swap(table);
                for (PyObject* q : old)
                    if (q) *slot(q) = q;
            }
            PyObject** at = slot(p);
            if (*at) {
                count--;
                return false;
            }
            *at = p;
            return true;
        }
        PyObject** slot(PyObject* p) {
            size_t h = (reinterpret_cast<uintptr_t>(p) >> 4) * 0x9e3779b97f4a7c15ull >> 20;
            while (table[h & (table.size() - 1)] && table[h & (table.size() - 1)] != p) h++;
            return &table[h & (table.size() - 1)];
        }
    };
    struct Param {
        size_t at, length;   // its name in `text`
        PyObject* object;    // borrowed: the module holds it
    };
    std::string text;
    Seen types, modules, seen;
    bool once;

    bool plain(PyObject* m) {
        struct Own { PyObject *name, *function; };   // what walks a module, as torch.nn.Module has it
        static const std::array<Own, 3> own = []() {
            std::array<Own, 3> a;
            const py::object base = py::module_::import("torch.nn").attr("Module");
            const char* const names[3] = {"named_modules", "named_parameters", "_named_members"};
            for (int i = 0; i < 3; i++) a[i] = Own{PyUnicode_InternFromString(names[i]), py::object(base.attr(names[i])).release().ptr()};
            return a;
        }();
        PyObject* const type = reinterpret_cast<PyObject*>(Py_TYPE(m));
        if (!types.insert(type)) return true;
        for (const Own& o : own) {
            const py::object f = py::reinterpret_steal<py::object>(PyObject_GetAttr(type, o.name));
            if (!f) PyErr_Clear();
            if (f.ptr() != o.function) return false;
        }
        return true;
    }

    bool visit(PyObject* m, std::string& prefix) {
        static PyObject* const s_params = PyUnicode_InternFromString("_parameters");
        static PyObject* const s_modules = PyUnicode_InternFromString("_modules");
        if (!modules.insert(m)) return true;
        if (!plain(m)) return false;
        const py::object ps = py::reinterpret_steal<py::object>(PyObject_GetAttr(m, s_params)),
                         ms = py::reinterpret_steal<py::object>(PyObject_GetAttr(m, s_modules));
        if (!ps || !ms || !PyDict_Check(ps.ptr()) || !PyDict_Check(ms.ptr())) {
            PyErr_Clear();
            return false;
        }
        PyObject *key, *value;
        Py_ssize_t at = 0, n = 0;
        while (PyDict_Next(ps.ptr(), &at, &key, &value)) {
            if (value == Py_None || (once && !seen.insert(value))) continue;
            const char* name = PyUnicode_AsUTF8AndSize(key, &n);
            if (!name || !THPVariable_CheckTypeExact(Py_TYPE(value))) return false;   // a Tensor or a Parameter, no other kind
            params.push_back({text.size(), prefix.size() + n, value});
            text.append(prefix).append(name, n);
        }
        const size_t length = prefix.size();
        at = 0;
        while (PyDict_Next(ms.ptr(), &at, &key, &value)) {
            if (value == Py_None) continue;
            const char* name = PyUnicode_AsUTF8AndSize(key, &n);
            if (!name) return false;
            prefix.append(name, n).push_back('.');
            const bool ok = visit(value, prefix);
            prefix.resize(length);
            if (!ok) return false;
        }
        return true;
    }

public:
    std::vector<Param> params;
    bool complete;
    Named(const py::object& root, bool once_) : once(once_) {
        params.reserve(256);
        text.reserve(16384);
        std::string prefix;
        complete = visit(root.ptr(), prefix);
        PyErr_Clear();
    }
    std::string_view name(const Param& p) const { return std::string_view(text).substr(p.at, p.length); }
    static const at::Tensor& tensor(const Param& p) { return THPVariable_Unpack(p.object); }
};

// A fingerprint under way on a stream: a kernel writes its value to pinned host memory.  The host allocator knows nothing
// of that kernel and hands the memory out again as soon as the tensor is gone, so whoever drops a fingerprint that
// nobody has read waits for the stream first.
class Fingerprint {
    torch::Tensor host;
    c10::hip::HIPStreamMasqueradingAsCUDA stream;
    bool pending = true;

public:
    explicit Fingerprint(c10::hip::HIPStreamMasqueradingAsCUDA s)
        : host(at::empty({1}, at::TensorOptions().dtype(torch::kDouble).pinned_memory(true))), stream(s) {}
    Fingerprint(Fingerprint&& o) noexcept : host(std::move(o.host)), stream(o.stream), pending(std::exchange(o.pending, false)) {}
    Fingerprint(const Fingerprint&) = delete;
    Fingerprint& operator=(const Fingerprint&) = delete;
    ~Fingerprint() {
        if (!pending) return;
        try {
            py::gil_scoped_release no_gil;
            stream.synchronize();
        } catch (...) {   // the stream is in error: the memory is not given back
            new torch::Tensor(std::move(host));
        }
    }
    double* out() { return static_cast<double*>(host.data_ptr()); }
    double value() {
        {
            py::gil_scoped_release no_gil;
            stream.synchronize();
        }
        pending = false;
        return *out();
    }
};

// sync.weight_fingerprint of a module, queued on the current stream of its parameters' device; None where they are not
// all fp32, contiguous and on one GPU, or the module is not walked as torch.nn.Module walks it
c10::optional<Fingerprint> fingerprint(const py::object& net) {
    Named named(net, true);
    if (!named.complete || named.params.empty()) return c10::nullopt;
    std::sort(named.params.begin(), named.params.end(), [&](const auto& a, const auto& b) { return named.name(a) < named.name(b); });
    std::vector<const float*> ptrs;
    std::vector<int64_t> numel;
    const c10::Device dev = Named::tensor(named.params[0]).device();
    ptrs.reserve(named.params.size());
    numel.reserve(named.params.size());
    for (const auto& np : named.params) {
        const at::Tensor& t = Named::tensor(np);
        if (!t.is_cuda() || t.device() != dev || t.scalar_type() != torch::kFloat || !t.is_contiguous() || !t.numel()) return c10::nullopt;
        ptrs.push_back(static_cast<const float*>(t.data_ptr()));
        numel.push_back(t.numel());
    }
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dev);
    const int n = (int)ptrs.size();
    const torch::Tensor partials = fresh({bf_fingerprint_partials(numel.data(), n)}, torch::kDouble);
    const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index());
    c10::optional<Fingerprint> f(std::in_place, stream);
    const int rc = bf_fingerprint(ptrs.data(), numel.data(), n, static_cast<double*>(partials.data_ptr()), f->out(), stream.stream());
    TORCH_CHECK(rc == BF_OK, "bf_fingerprint failed (", rc, "): ", bf_last_error());
    return f;
}

// pack_board of a whole network, its parameters found by name; None where one is missing under its name
c10::optional<std::pair<torch::Tensor, torch::Tensor>> pack_net(const py::object& net, int64_t d_model, int64_t n_layers, int64_t d_ff,
                                                                int64_t n_value, double eps, bool fp8, int64_t device) {
    static const char* const of_layer[12] = {"norm1.weight", "norm1.bias", "self_attn.in_proj_weight", "self_attn.in_proj_bias",
                                             "self_attn.out_proj.weight", "self_attn.out_proj.bias", "norm2.weight", "norm2.bias",
                                             "linear1.weight", "linear1.bias", "linear2.weight", "linear2.bias"};
    static const char* const of_net[10] = {"emb_square.weight", "emb_type_special.weight", "emb_color_turn.weight", "emb_clock.weight",
                                           "emb_rep.weight", "norm_f.weight", "norm_f.bias", "policy.weight", "promo.weight", "value.weight"};
    Named named(net, false);
    if (!named.complete) return c10::nullopt;
    std::sort(named.params.begin(), named.params.end(), [&](const auto& a, const auto& b) { return named.name(a) < named.name(b); });
    std::vector<torch::Tensor> params;
    params.reserve(12 * n_layers + 10);
    auto take = [&](std::string_view name) {
        const auto it = std::lower_bound(named.params.begin(), named.params.end(), name, [&](const auto& a, std::string_view b) { return named.name(a) < b; });
        if (it == named.params.end() || named.name(*it) != name) return false;
        params.push_back(Named::tensor(*it));
        return true;
    };
    for (int64_t i = 0; i < n_layers; i++) {
        std::string name = "encoder.layers." + std::to_string(i) + ".";
        const size_t length = name.size();
        for (const char* part : of_layer) {
            if (!take(name.append(part))) return c10::nullopt;
            name.resize(length);
        }
    }
    for (const char* name : of_net)
        if (!take(name)) return c10::nullopt;
    return pack_board(params, d_model, n_layers, d_ff, n_value, eps, fp8, device);
}

// Cycles per phase summed over the wavefronts of one launch of the profiling build (see
// bf_profile_phases); returns an int64 tensor on the device, already written when it is read.
torch::Tensor profile_phases(torch::Tensor boards, torch::Tensor control, torch::Tensor rep, torch::Tensor weights,
                             torch::Tensor params, torch::Tensor policy, torch::Tensor promo, torch::Tensor value,
                             int64_t d_model, int64_t n_layers, int64_t n_heads, int64_t d_ff, double eps, int64_t kernel,
                             int64_t n_value, int64_t vmode, OptTensor mask, OptTensor best_move, OptTensor workspace) {
    const Checked c = check(boards, control, rep, weights, params, policy, promo, value, d_model, n_layers, n_heads,
                            d_ff, eps, BF_QUANT_INT8, kernel, n_value, vmode, mask, best_move, c10::nullopt, workspace);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(c.device);
    auto cycles = torch::zeros({(int64_t)bf_profile_phase_count()}, torch::dtype(torch::kLong).device(c.device));
    const int rc = bf_profile_phases(&c.a, c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(c.device.index()).stream(),
                                     reinterpret_cast<uint64_t*>(cycles.data_ptr<int64_t>()));
    TORCH_CHECK(rc == BF_OK, "bf_profile_phases failed (", rc, "): ", bf_last_error());
    return cycles;
}

// ---- the two calls a search makes every step, as plain vector calls ---------------------------------
// Positional arguments straight from the interpreter's stack and results wrapped here: pybind11's dispatch and casters
// are 0.4 us of a 4 us call.
const torch::Tensor& tensor_arg(PyObject* o) {
    if (!THPVariable_Check(o)) throw py::type_error("expected a tensor");
    return THPVariable_Unpack(o);
}
OptTensor opt_tensor_arg(PyObject* o) {
    if (o == Py_None) return c10::nullopt;
    return tensor_arg(o);
}
c10::optional<std::pair<torch::Tensor, torch::Tensor>> opt_pair_arg(PyObject* o) {
    if (o == Py_None) return c10::nullopt;
    const py::object two = py::reinterpret_steal<py::object>(PySequence_Fast(o, "expected a pair of tensors"));
    if (!two) throw py::error_already_set();
    if (PySequence_Fast_GET_SIZE(two.ptr()) != 2) throw py::type_error("expected a pair of tensors");
    return std::pair<torch::Tensor, torch::Tensor>(tensor_arg(PySequence_Fast_GET_ITEM(two.ptr(), 0)), tensor_arg(PySequence_Fast_GET_ITEM(two.ptr(), 1)));
}
template <typename F>
PyObject* guarded(Py_ssize_t got, Py_ssize_t want, const F& body) {
    try {
        if (got != want) throw py::type_error(c10::str("expected ", want, " positional arguments, got ", got));
        return body();
    } catch (py::error_already_set& e) {
        e.restore();
    } catch (const py::builtin_exception& e) {
        e.set_error();
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}
PyObject* call_movegen(PyObject*, PyObject* const* a, Py_ssize_t n) {   // boards, control, out
    return guarded(n, 3, [&]() -> PyObject* {
        const auto r = movegen(tensor_arg(a[0]), tensor_arg(a[1]), opt_pair_arg(a[2]));
        const py::object t = py::reinterpret_steal<py::object>(PyTuple_New(2));
        if (!t) throw py::error_already_set();
        PyTuple_SET_ITEM(t.ptr(), 0, THPVariable_Wrap(r.first));
        PyTuple_SET_ITEM(t.ptr(), 1, THPVariable_Wrap(r.second));
        return t.inc_ref().ptr();
    });
}
PyObject* call_expand_edges(PyObject*, PyObject* const* a, Py_ssize_t n) {   // as expand_edges
    return guarded(n, 10, [&]() -> PyObject* {
        const long edges = PyLong_AsLong(a[6]);
        if (edges == -1 && PyErr_Occurred()) throw py::error_already_set();
        c10::optional<py::dict> out;
        if (a[8] != Py_None) out = py::reinterpret_borrow<py::object>(a[8]).cast<py::dict>();
        return expand_edges(tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]), tensor_arg(a[4]), tensor_arg(a[5]), edges,
                            opt_tensor_arg(a[7]), out, opt_pair_arg(a[9])).release().ptr();
    });
}
PyObject* call_movegen_expand(PyObject*, PyObject* const* a, Py_ssize_t n) {   // as movegen_expand
    return guarded(n, 7, [&]() -> PyObject* {
        const long edges = PyLong_AsLong(a[5]);
        if (edges == -1 && PyErr_Occurred()) throw py::error_already_set();
        c10::optional<py::dict> out;
        if (a[6] != Py_None) out = py::reinterpret_borrow<py::object>(a[6]).cast<py::dict>();
        return movegen_expand(tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]), tensor_arg(a[4]), edges, out).release().ptr();
    });
}
PyMethodDef vector_calls[] = {
    {"movegen", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&call_movegen)), METH_FASTCALL, "(boards, control, out) -> legal-move words and check flags"},
    {"expand_edges", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&call_expand_edges)), METH_FASTCALL,
     "(policy, promo, value, mask, boards, control, max_edges, active, out, leaves) -> edges of search nodes"},
    {"movegen_expand", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&call_movegen_expand)), METH_FASTCALL,
     "(policy, promo, value, boards, control, max_edges, out) -> edges of search nodes, legal-move words and check flags"},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "MI355X evaluator: torch tensors in, one launch on the current HIP stream";
    m.def("model_forward", &model_forward, "boards in, policy / promo / value out", py::arg("boards"), py::arg("control"),
          py::arg("rep"), py::arg("weights"), py::arg("params"), py::arg("policy"), py::arg("promo"), py::arg("value"),
          py::arg("d_model"), py::arg("n_layers"), py::arg("n_heads"), py::arg("d_ff"), py::arg("eps"),
          py::arg("quant") = 0, py::arg("kernel") = 0, py::arg("n_value") = 1, py::arg("vmode") = 0,
          py::arg("mask") = py::none(), py::arg("best_move") = py::none(), py::arg("active") = py::none(),
          py::arg("workspace") = py::none(), py::arg("leaf_index") = py::none(), py::arg("leaf_count") = py::none(),
          py::arg("team_workspace") = py::none());
    m.def("encoder_forward", &encoder_forward, "the encoder stack alone, in place on y", py::arg("y"), py::arg("weights"),
          py::arg("params"), py::arg("alive"), py::arg("d_model"), py::arg("n_layers"), py::arg("n_heads"), py::arg("d_ff"),
          py::arg("eps"), py::arg("quant") = 0, py::arg("kernel") = 0, py::arg("n_value") = 1, py::arg("workspace") = py::none());
    if (PyModule_AddFunctions(m.ptr(), vector_calls)) throw py::error_already_set();
    m.def("compact_leaves", &compact_leaves, "leaf flags to an ordered list and its length", py::arg("flags"), py::arg("out") = py::none());
    m.def("pack_board", &pack_board, "a network's parameters into the board blobs", py::arg("params"), py::arg("d_model"), py::arg("n_layers"),
          py::arg("d_ff"), py::arg("n_value"), py::arg("eps"), py::arg("fp8"), py::arg("device"));
    m.def("pack_net", &pack_net, "the same for a whole network, or None where its parameters have other names", py::arg("net"), py::arg("d_model"),
          py::arg("n_layers"), py::arg("d_ff"), py::arg("n_value"), py::arg("eps"), py::arg("fp8"), py::arg("device"));
    py::class_<Fingerprint>(m, "Fingerprint").def("value", &Fingerprint::value, "the sum, once the stream has come to it");
    m.def("fingerprint", &fingerprint, "index-weighted float64 sum over a module's parameters on one GPU, queued, or None", py::arg("net"));
    m.def("profile_phases", &profile_phases, "cycles per phase of one profiled launch", py::arg("boards"),
          py::arg("control"), py::arg("rep"), py::arg("weights"), py::arg("params"), py::arg("policy"), py::arg("promo"),
          py::arg("value"), py::arg("d_model"), py::arg("n_layers"), py::arg("n_heads"), py::arg("d_ff"), py::arg("eps"),
          py::arg("kernel") = 0, py::arg("n_value") = 1, py::arg("vmode") = 0, py::arg("mask") = py::none(),
          py::arg("best_move") = py::none(), py::arg("workspace") = py::none());
    m.def("profile_phase_names", []() {
        std::vector<std::string> names;
        for (int i = 0; i < bf_profile_phase_count(); i++) names.emplace_back(bf_profile_phase_name(i));
        return names;
    }, "phase names, in slot order");
    m.def("int8_q_max", []() {
        double s8 = 0.0, u8 = 0.0;
        bf_int8_q_max(&s8, &u8);
        return std::pair<double, double>{s8, u8};
    }, "the s8 and u8 quantisation maxima compiled into the library");
    m.def("fp8_q_max", []() { return bf_fp8_q_max(); }, "what a row's largest magnitude maps to in e4m3");
    m.def("abi_tag", []() { return (uint64_t)BF_ABI_TAG; }, "interface tag of the header this module was compiled against");
    m.def("library_abi_tag", []() { return bf_abi_tag(); }, "interface tag of the library this module is linked to");
    m.def("kernel_choice", [](int64_t d_model, int64_t n_layers, int64_t n_heads, int64_t d_ff, int64_t n_value, int64_t n,
                              int64_t quant, int64_t kernel, bool board_blobs) {
        bf_eval_args a{};
        a.shape = bf_shape{(int32_t)d_model, (int32_t)n_layers, (int32_t)n_heads, (int32_t)d_ff, (int32_t)n_value, 1e-5f};
        a.n = n;
        a.quant = (int32_t)quant;
        a.kernel = (int32_t)kernel;
        const auto nonnull = reinterpret_cast<const uint8_t*>(uintptr_t(16));     // only tested for NULL
        if (board_blobs) { a.board_wstream = nonnull; a.board_fparams = reinterpret_cast<const float*>(nonnull); }
        else { a.wstream = nonnull; a.fparams = reinterpret_cast<const float*>(nonnull); }
        const int rc = bf_kernel_choice(&a);
        TORCH_CHECK(rc >= 0, "bf_kernel_choice failed (", rc, "): ", bf_last_error());
        return rc;
    }, "the kernel (enum bf_kernel) these arguments name or, for AUTO, whose launches they are");
}
