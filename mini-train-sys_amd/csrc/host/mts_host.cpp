// Host path of the `hip` backend: contract checks, allocation and the autograd nodes of the operators, in front of the C ABI
// of the kernel library (include/mts_moe.h).
//
// A layer step is seven to nine launches, 60 to 350 us of kernels at up to 5000 tokens.  Allocating two dozen tensors,
// marshalling two hundred arguments and passing the interpreter lock between the caller's thread and autograd's took 220 to
// 360 us in Python (two speeds, from process to process), so that every small call ran at the speed of the host.  Native, a
// forward pass of 16 tokens takes 48 us instead of 102 (its five kernels: 35) and a training step of 512 tokens 145 to 185, by
// box, instead of 220 to 360 (its eight kernels: 112): the host still sets the time of both.
//
// Nothing here synchronises with the GPU.  Every buffer is a torch tensor from the caching allocator; the backward pass of
// the operator forks two side streams for kernels that do not depend on one another and joins them before it returns.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <cmath>
#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "mts_moe.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
typedef std::optional<Tensor> MaybeTensor;

// ---- small helpers ---------------------------------------------------------------------------------------------------------

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
template <typename T>
T* ptr_as(const Tensor& t) { return static_cast<T*>(ptr(t)); }

void check(int code, const char* what) { TORCH_CHECK(code == 0, what, " failed: ", mts_error_string(code), " (code ", code, ")"); }

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kBFloat16: return MTS_BF16;
        case at::kHalf: return MTS_F16;
        case at::kFloat: return MTS_F32;
        default: TORCH_CHECK(false, "unsupported dtype ", t);
    }
}
int dtype_code(const Tensor& t) { return dtype_code(t.scalar_type()); }
bool is_activation_type(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf || t == at::kFloat; }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor bytes(int64_t n, const Tensor& like) { return at::empty({n > 4 ? n : 4}, like.options().dtype(at::kByte)); }
Tensor f32(at::IntArrayRef size, const Tensor& like) { return at::empty(size, like.options().dtype(at::kFloat)); }
Tensor i32(at::IntArrayRef size, const Tensor& like) { return at::empty(size, like.options().dtype(at::kInt)); }
Tensor like_f32(const Tensor& g) { return g.defined() ? g.to(at::kFloat).contiguous() : g; }
bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
Tensor dense16(const Tensor& t) {   // dense and starting on a 16-byte boundary (a view may start inside an allocation)
    Tensor d = t.contiguous();
    return aligned16(d) ? d : d.clone();
}
// Whether a kernel may be run on the tensors' memory in the place of stock operators: not where those are looked at by a
// function transform (vmap, grad, forward mode), a trace, a dispatch mode or a subclass.
bool nobody_dispatches() {
    using c10::DispatchKey;
    return !c10::impl::tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !c10::impl::tls_is_dispatch_key_included(DispatchKey::Tracer) && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}
bool is_plain(const Tensor& t) {
    using c10::DispatchKey;
    static const c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::Batched, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                              DispatchKey::Functionalize, DispatchKey::Conjugate, DispatchKey::Negative, DispatchKey::ZeroTensor});
    return !t.key_set().has_any(wrapped) && !t._fw_grad(/*level=*/0).defined();
}
template <typename... Ts>
bool all_plain(const Ts&... t) {
    return nobody_dispatches() && !at::impl::torch_function_mode_enabled() && (is_plain(t) && ...);
}
// Whether a backward pass is written out in stock operators: its gradients are themselves to be differentiated (create_graph),
// they come batched or wrapped (is_grads_batched, vmap over autograd.grad), or somebody looks on.
bool written_out(const variable_list& grads) {
    if (at::GradMode::is_enabled() || !nobody_dispatches()) return true;
    for (const Tensor& g : grads)
        if (g.defined() && !is_plain(g)) return true;
    return false;
}
template <typename... Ts>
bool on_one_gpu(const Tensor& first, const Ts&... others) {
    return first.is_cuda() && ((others.device() == first.device()) && ...);
}

// Contiguous elements of `base`, a dense allocation of bytes, as a tensor of their own.  No view: the parts of an allocation do not overlap, and
// none of those made this way is handed to a caller who could differentiate through it.
Tensor part_of(const Tensor& base, int64_t first_byte, at::IntArrayRef size, at::ScalarType type) {
    auto impl = c10::make_intrusive<c10::TensorImpl>(c10::Storage(base.storage()), base.key_set(), c10::scalarTypeToTypeMeta(type));
    impl->set_storage_offset(base.storage_offset() + first_byte / (int64_t)c10::elementSize(type));
    impl->set_sizes_contiguous(size);
    return Tensor(std::move(impl));
}

// Tensors of one call that come and go together, in one allocation where that is small: a call of few tokens is bound by the host, which
// spends about a microsecond on each allocation and on each view (16 tokens 768/1024: a call without gradients 48 -> 36 us, 512 tokens with them 165 -> 137).  Above the limit each
// has its own, so that no block grows with the sum of the large ones.
class Together {
    static constexpr int64_t kMostBytes = 32 << 20;
    struct Job {
        Tensor* out;
        std::array<int64_t, 2> size;
        int dims;
        at::ScalarType type;
        int64_t bytes() const { return (size[0] * (dims > 1 ? size[1] : 1) * (int64_t)c10::elementSize(type) + 255) / 256 * 256; }
        at::IntArrayRef sizes() const { return at::IntArrayRef(size.data(), (size_t)dims); }
    };
    c10::SmallVector<Job, 12> jobs_;
    const Tensor& like_;

public:
    explicit Together(const Tensor& like) : like_(like) {}
    void add(Tensor& out, int64_t rows, int64_t columns, at::ScalarType type) { jobs_.push_back({&out, {rows, columns}, 2, type}); }
    void add(Tensor& out, int64_t count, at::ScalarType type) { jobs_.push_back({&out, {count, 1}, 1, type}); }
    void make() {
        int64_t total = 0;
        for (const Job& j : jobs_) total += j.bytes();
        if (total > kMostBytes || jobs_.size() < 2) {
            for (const Job& j : jobs_) *j.out = at::empty(j.sizes(), like_.options().dtype(j.type));
            return;
        }
        const Tensor base = at::empty({total}, like_.options().dtype(at::kByte));
        int64_t at_byte = 0;
        for (const Job& j : jobs_) {
            *j.out = part_of(base, at_byte, j.sizes(), j.type);
            at_byte += j.bytes();
        }
    }
};

// ---- contracts ---------------------------------------------------------------------------------------------------------------
// The first requirement that the arguments miss, or NULL.

constexpr int64_t kMaxExperts = MTS_MAX_MOE_EXPERTS, kMaxTopK = MTS_MAX_TOP_K, kMaxRouterExperts = MTS_MAX_EXPERTS;
constexpr int64_t k2GiB = 1LL << 31;

const char* expert_violation(const Tensor& x, const Tensor& w1, const Tensor& w2) {
    if (x.dim() != 2 || w1.dim() != 3 || w2.dim() != 3) return "x is [T,H], gate_up_proj [E,2I,H] and down_proj [E,H,I]";
    const int64_t T = x.size(0), H = x.size(1), E = w1.size(0), two_i = w1.size(1), I = two_i / 2;
    if (!on_one_gpu(x, w1, w2)) return "all tensors on one GPU";
    const auto t = x.scalar_type();
    if (!is_activation_type(t)) return "activations are bf16, fp16 or fp32";
    if (T <= 0) return "at least one token";
    if (E <= 0 || E > kMaxExperts) return "between 1 and 65534 experts";
    if (two_i % 2 || w1.size(2) != H || w2.size(0) != E || w2.size(1) != H || w2.size(2) != I)
        return "gate_up_proj is [E,2I,H] and down_proj [E,H,I] for x [T,H]";
    // expert parameters come in the activation dtype or as fp32 master weights; fp32 activations take 16-bit parameters as
    // well (widened once per call)
    auto fits = [&](at::ScalarType p) { return p == at::kFloat || p == t || (t == at::kFloat && is_activation_type(p)); };
    if (!fits(w1.scalar_type()) || !fits(w2.scalar_type()))
        return "expert parameters in the activation dtype or fp32 (any of fp32/bf16/fp16 under fp32 activations)";
    // rows of x and of dO are gathered from anywhere through 32-bit offsets; the [T*K, ...] intermediates are addressed tile
    // by tile and may be larger
    if (t != at::kFloat && (T * H * 2 >= k2GiB || 2 * I * H * 2 >= k2GiB)) return "16-bit activations and one expert's weights smaller than 2 GiB each";
    return nullptr;
}

const char* routing_violation(const Tensor& x, const Tensor& w1, const Tensor& index, const Tensor& weights) {
    if (index.dim() != 2) return "top_k_index is [T,K]";
    const int64_t K = index.size(1);
    if (!on_one_gpu(x, index, weights)) return "routing tensors on the activations' GPU";
    if (weights.sizes() != index.sizes() || index.size(0) != x.size(0)) return "top_k_index and top_k_weights are [T,K]";
    if (K <= 0 || K > std::min<int64_t>(w1.size(0), 32768)) return "1 <= K <= number of experts (at most 32768)";
    if (x.size(0) * K >= k2GiB) return "fewer than 2^31 routes";
    if (index.scalar_type() != at::kInt) return "int32 expert indices";
    if (weights.scalar_type() != x.scalar_type()) return "routing weights in the activation dtype";
    return nullptr;
}

const char* fused_moe_violation(const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& index, const Tensor& weights) {
    const char* missed = expert_violation(x, w1, w2);
    return missed ? missed : routing_violation(x, w1, index, weights);
}

// The kernels move 16 bytes per lane: rows are whole 16-byte chunks, or zero-padded to that by the caller.
bool needs_padding(const Tensor& x, const Tensor& w1) {
    const bool wide = x.scalar_type() == at::kFloat;
    return x.size(1) % (wide ? 4 : 8) != 0 || (!wide && (w1.size(1) / 2) % 8 != 0);
}

// Up to 16 experts the projection kernels keep W_r in LDS; more take the kernels on the fp32 matrix instruction.
constexpr int64_t kFewExperts = 16;
bool router_logits_supported(const Tensor& x, const Tensor& w) {
    return all_plain(x, w) && on_one_gpu(x, w) && x.dim() == 2 && w.dim() == 2 && is_activation_type(x.scalar_type()) &&
           w.scalar_type() == at::kFloat && x.size(0) > 0 && x.size(1) == w.size(1) &&
           (w.size(0) <= kFewExperts ? x.size(1) % 4 == 0 && x.size(1) <= 4096 && w.size(0) * w.size(1) * 4 <= 128 * 1024
                                     : mts_router_wide_supported(x.size(1), w.size(0)));
}

const char* layer_violation(const Tensor& x, const Tensor& w_r, const Tensor& w1, const Tensor& w2, int64_t top_k) {
    if (const char* missed = expert_violation(x, w1, w2)) return missed;
    const int64_t E = w1.size(0);
    if (w_r.dim() != 2 || w_r.size(0) != E) return "router weight is [E,H]";
    if (!router_logits_supported(x, w_r))
        return "an fp32 router weight on the same GPU, at most 1024 experts, and up to 16 of them a hidden size of at most 4096 (E * H <= 32768)";
    if (top_k < 1 || top_k > std::min(E, kMaxTopK)) return "1 <= top_k <= min(E, 8)";
    if (needs_padding(x, w1)) return "hidden and expert widths that are whole 16-byte chunks";
    if (x.size(0) * top_k >= k2GiB) return "fewer than 2^31 routes";
    return nullptr;
}

// ---- options -----------------------------------------------------------------------------------------------------------------

// Comparison switches of the Python side (kernels/hip/switches.py), as they stand when an operator is called.
enum Switch : int64_t { OVERLAP = 1, JOINT_BWD = 2, JOINT_FWD = 4, TAIL_IN_JOINT = 8, COMBINE_IN_TAIL = 16, JOINT_SCHEDULE = 32, WEIGHTED_POST = 64, NO_BACKWARD = 1 << 20 /* set here: nothing that this call computes will be differentiated */ };

struct Options {
    int64_t switches;
    int64_t dw_workspace_limit;   // row-chunk workspaces of the weight-gradient GEMMs beyond this size are done without
    bool on(Switch s) const { return (switches & s) != 0; }
};

template <typename... Ts>
int64_t no_backward(const Ts&... t) {
    return at::GradMode::is_enabled() && (t.requires_grad() || ...) ? 0 : NO_BACKWARD;
}

// Counters of the joint gate/up + down launch, owned by the Python side (one per device and stream): an object with
// before_launch(), get(bytes) and after_launch().  Forward passes run under the interpreter lock.
pybind11::object* joint_workspace_of = nullptr;   // device index -> that object; never destroyed

// ---- streams -----------------------------------------------------------------------------------------------------------------

hipStream_t side_stream(int device, int index) {
    static std::mutex lock;
    static std::map<std::pair<int, int>, c10::hip::HIPStream> streams;
    std::lock_guard<std::mutex> held(lock);
    auto it = streams.find({device, index});
    if (it == streams.end()) it = streams.emplace(std::make_pair(device, index), c10::hip::getStreamFromPool(/*isHighPriority=*/false, device)).first;
    return it->second.stream();
}

// work enqueued on `to` from here on waits for what `from` holds now
void order_after(hipStream_t to, hipStream_t from) {
    if (to == from) return;
    hipEvent_t ev;
    TORCH_CHECK(hipEventCreateWithFlags(&ev, hipEventDisableTiming) == hipSuccess, "hipEventCreate failed");
    const bool ok = hipEventRecord(ev, from) == hipSuccess && hipStreamWaitEvent(to, ev, 0) == hipSuccess;
    (void)hipEventDestroy(ev);   // released once the recorded work has passed it
    TORCH_CHECK(ok, "ordering two streams failed");
}

// Side streams that work has been forked onto.  The caller's stream waits for them before what they read and write is released,
// also where an error (a refused call, memory that runs out) leaves the function: the allocator knows the caller's stream only.
class Forked {
    hipStream_t main_, streams_[2] = {};
    int n_ = 0;

  public:
    explicit Forked(hipStream_t main) : main_(main) {}
    Forked(const Forked&) = delete;
    void fork(hipStream_t s) {
        if (s == main_) return;
        if (s != streams_[0] && s != streams_[1]) streams_[n_++] = s;
        order_after(s, main_);
    }
    // The longest comes last (dW1): a wait costs the caller's stream some 5 us of its own, which the waits before the last one
    // spend while the last one's work still runs.
    void join() {
        for (int i = 0; i < n_; ++i) order_after(main_, streams_[i]);
        n_ = 0;
    }
    ~Forked() {
        try {
            join();
        } catch (...) {   // on top of the error that is under way
        }
    }
};

// ---- experts: forward and backward ---------------------------------------------------------------------------------------------

struct Routing {
    Tensor expert_start, x_gather, s_scatter, s_reverse;
};

// Routing metadata of given expert indices (the per-row arrays start on 16-byte boundaries).
Routing route(const Tensor& index, int64_t E) {
    const int64_t T = index.size(0), K = index.size(1), TK = T * K, ws_bytes = mts_moe_route_workspace_bytes(T, K, E);
    Tensor counts, ws;
    Routing r;
    Together together(index);
    together.add(counts, E, at::kInt);
    together.add(r.expert_start, E + 1, at::kInt);
    together.add(r.s_scatter, TK, at::kInt);
    together.add(r.s_reverse, TK, at::kInt);
    together.add(r.x_gather, TK, at::kInt);
    together.add(ws, std::max<int64_t>(ws_bytes, 4), at::kByte);
    together.make();
    check(mts_moe_route(ptr_as<int32_t>(index), T, K, E, 64, ptr_as<int32_t>(counts), ptr_as<int32_t>(r.expert_start), ptr_as<int32_t>(r.s_scatter),
                        ptr_as<int32_t>(r.s_reverse), ptr_as<int32_t>(r.x_gather), nullptr, nullptr, nullptr, ptr(ws), ws_bytes, stream_of(index)),
          "mts_moe_route");
    return r;
}

// Copy of an expert weight [E,R,C] in the activation dtype, optionally as [E,C,R].
Tensor stage(const Tensor& w, bool transpose, at::ScalarType dtype, void* stream) {
    if (!transpose && w.scalar_type() == dtype) return w;
    const int64_t E = w.size(0), R = w.size(1), C = w.size(2);
    Tensor out = at::empty({E, transpose ? C : R, transpose ? R : C}, w.options().dtype(dtype));
    check(mts_moe_stage_weights(ptr(w), dtype_code(w), ptr(out), dtype_code(dtype), E, R, C, transpose, stream), "mts_moe_stage_weights");
    return out;
}

// How the backward GEMMs are told that a weight comes as it is stored; 0: they need a transposed copy.
int stored_layout(int act, int64_t H, int64_t I) { return act == MTS_F32 ? MTS_STORED_F32 : mts_moe_bwd_weights_as_stored(act, H, I); }

// What the forward pass leaves for the backward pass.  The tensors travel through save_for_backward in this order.
struct Saved {
    Tensor x, w1, w2, pre_act, weights, expert_start, x_gather, s_scatter, s_reverse, post_act, staged1, staged2;
    static constexpr size_t kCount = 12;
    void append_to(variable_list& v) const {
        v.insert(v.end(), {x, w1, w2, pre_act, weights, expert_start, x_gather, s_scatter, s_reverse, post_act, staged1, staged2});
    }
    explicit Saved(const variable_list& v)
        : x(v[0]), w1(v[1]), w2(v[2]), pre_act(v[3]), weights(v[4]), expert_start(v[5]), x_gather(v[6]), s_scatter(v[7]), s_reverse(v[8]),
          post_act(v[9]), staged1(v[10]), staged2(v[11]) {}
    Saved() = default;
};

bool masters(const Tensor& x, const Tensor& w1, const Tensor& w2) {
    return w1.scalar_type() == at::kFloat && w2.scalar_type() == at::kFloat && x.scalar_type() != at::kFloat;
}
// With few rows the kernels read the weights once and round fp32 ones themselves; a backward pass wants the rounded copies.  `ride`: these would be made
// beside the head.
bool reads_masters(const Tensor& x, const Tensor& w1, const Tensor& w2, int64_t TK, const Options& opt, bool ride = false) {
    if (!masters(x, w1, w2) || !opt.on(NO_BACKWARD)) return false;
    const int act = dtype_code(x);
    const int64_t T = x.size(0), E = w1.size(0), H = x.size(1), I = w1.size(1) / 2;
    return ride ? mts_moe_fwd_few_rows_preferred_to_ride(act, T, TK, E, H, I) : mts_moe_fwd_few_rows_preferred(act, MTS_F32, T, TK, E, H, I);
}
// fp32 master weights that can be rounded together (the backward pass reuses the copies)
bool copies_masters(const Tensor& x, const Tensor& w1, const Tensor& w2) { return masters(x, w1, w2) && w1.numel() % 8 == 0 && w2.numel() % 8 == 0; }

// The expert weights as the forward kernels read them: as they are, or copies in the activation dtype.
std::pair<Tensor, Tensor> forward_weights(const Tensor& x, const Tensor& w1, const Tensor& w2, int64_t TK, const Options& opt) {
    if (reads_masters(x, w1, w2, TK, opt)) return {w1, w2};
    void* stream = stream_of(x);
    if (!copies_masters(x, w1, w2)) return {stage(w1, false, x.scalar_type(), stream), stage(w2, false, x.scalar_type(), stream)};
    Tensor copy1 = at::empty(w1.sizes(), x.options()), copy2 = at::empty(w2.sizes(), x.options());
    check(mts_moe_cast_weights_pair(ptr_as<float>(w1), ptr(copy1), w1.numel(), ptr_as<float>(w2), ptr(copy2), w2.numel(), dtype_code(x), stream),
          "mts_moe_cast_weights_pair");
    return {copy1, copy2};
}

// What the backward pass of a forward pass needs; `w1`, `w2`: the weights that the kernels read, kept where they are copies that the backward GEMMs take.
void keep(Saved& s, const Tensor& x, const Tensor& w1_in, const Tensor& w2_in, const Tensor& w1, const Tensor& w2, const Tensor& pre_act, const Tensor& post_act,
          const Tensor& weights, const Routing& r) {
    s.x = x, s.w1 = w1_in, s.w2 = w2_in, s.pre_act = pre_act, s.post_act = post_act, s.weights = weights;
    s.expert_start = r.expert_start, s.x_gather = r.x_gather, s.s_scatter = r.s_scatter, s.s_reverse = r.s_reverse;
    if (stored_layout(dtype_code(x), x.size(1), w1_in.size(1) / 2)) {   // the backward GEMMs read the weights as stored: they reuse casts made here
        if (!w1.is_same(w1_in)) s.staged1 = w1;
        if (!w2.is_same(w2_in)) s.staged2 = w2;
    }
}

// Gate/up + SwiGLU, down projection and combine for routes that are already sorted.  `weights`: flat, activation dtype.
// `post_act` [TK,I] and `y` [TK,H]: scratch that the caller has, or undefined; `w1`, `w2`: copies of master weights that the caller has made
Tensor experts_forward(const Tensor& x, const Tensor& w1_in, const Tensor& w2_in, const Tensor& weights, const Routing& r, const Options& opt, Saved& s,
                       Tensor post_act = Tensor(), Tensor y = Tensor(), Tensor w1 = Tensor(), Tensor w2 = Tensor()) {
    const int64_t T = x.size(0), H = x.size(1), E = w1_in.size(0), I = w1_in.size(1) / 2, TK = weights.numel(), K = TK / T;
    const auto dtype = x.scalar_type();
    const int act = dtype_code(dtype);
    void* stream = stream_of(x);
    const bool weighted = opt.on(WEIGHTED_POST);
    if (!w1.defined()) std::tie(w1, w2) = forward_weights(x, w1_in, w2_in, TK, opt);
    const bool few = (dtype != at::kFloat && dtype_code(w1) == MTS_F32) || mts_moe_fwd_few_rows_preferred(act, act, T, TK, E, H, I);
    // The routing weight is applied where the activation is formed: post_act = s * silu(g) * u.  The down projection then
    // yields s * y, the combine is a plain sum, and post_act is at the same time the operand of the dW2 GEMM, so it is kept
    // for the backward pass instead of being written again there.
    Tensor pre_act;
    if (!post_act.defined()) post_act = at::empty({TK, I}, x.options());
    if (!y.defined()) y = at::empty({TK, H}, x.options());
    if (!opt.on(NO_BACKWARD) || dtype == at::kFloat) pre_act = at::empty({TK, 2 * I}, x.options());
    void* route_w = weighted ? ptr(weights) : nullptr;
    int32_t* route_entry = weighted ? ptr_as<int32_t>(r.s_scatter) : nullptr;
    if (few) {
        check(mts_moe_fwd_few_rows(ptr(x), ptr(w1), ptr(w2), dtype_code(w1), ptr_as<int32_t>(r.x_gather), ptr_as<int32_t>(r.expert_start), route_w, route_entry,
                                   T, K, E, H, I, act, ptr(pre_act), ptr(post_act), ptr(y), stream),
              "mts_moe_fwd_few_rows");
    } else if (opt.on(JOINT_FWD) && mts_moe_fwd_joint_preferred(act, TK, E, H, I)) {
        // one launch: the down tiles take the CUs as the gate/up tiles leave them
        const int64_t need = mts_moe_fwd_joint_workspace_bytes(TK, E);
        pybind11::object ws = (*joint_workspace_of)((int)x.device().index());
        ws.attr("before_launch")();
        Tensor counters = ws.attr("get")(need).cast<Tensor>();
        check(mts_moe_fwd_gateup_down(ptr(x), ptr(w1), ptr(w2), ptr_as<int32_t>(r.x_gather), ptr_as<int32_t>(r.expert_start), route_w, route_entry, T, K, E, H,
                                      I, act, ptr(pre_act), ptr(post_act), ptr(y), ptr_as<int32_t>(counters), need, stream),
              "mts_moe_fwd_gateup_down");
        ws.attr("after_launch")();
    } else {
        check(mts_moe_fwd_gateup_swiglu(ptr(x), ptr(w1), ptr_as<int32_t>(r.x_gather), ptr_as<int32_t>(r.expert_start), route_w, route_entry, T, K, E, H, I,
                                        act, ptr(pre_act), ptr(post_act), stream),
              "mts_moe_fwd_gateup_swiglu");
        check(mts_moe_fwd_down(ptr(post_act), ptr(w2), ptr_as<int32_t>(r.expert_start), TK, E, H, I, act, ptr(y), stream), "mts_moe_fwd_down");
    }
    Tensor out = at::empty({T, H}, x.options());
    check(mts_moe_combine(ptr(y), weighted ? nullptr : ptr(weights), nullptr, ptr_as<int32_t>(r.s_reverse), T, K, H, act, ptr(out), stream), "mts_moe_combine");
    keep(s, x, w1_in, w2_in, w1, w2, pre_act, weighted ? post_act : Tensor(), weights, r);
    return out;
}

struct Needs {
    bool x, w1, w2, s;
};

// The router's side of the path from x to the loss, for a caller that owns it (the layer node): its gradient of x is added
// inside the dX combine, and where the one-launch backward applies its kernels ride in that launch.
struct RouterTail {
    Tensor w_r, logits, weights, indices, counts, g_prob_mean, g_z_loss, g_load_balance;
    bool normalize;
    Tensor kept_reverse;   // defined: the weights were limited to the routes it gives a row, and renormalised
    Tensor dx_r, dw_r;     // results
};

struct ExpertGrads {
    Tensor dx, dw1, dw2, ds;
};

// The projection of many experts stands in for a library product that takes any alignment.
Tensor dense_router_operand(const Tensor& t, int64_t E) { return E > kFewExperts ? dense16(t) : t.contiguous(); }

void router_projection_forward(const Tensor& x, const Tensor& w, const Tensor& logits) {
    const int64_t T = x.size(0), H = x.size(1), E = w.size(0);
    if (E > kFewExperts)
        check(mts_router_wide_fwd(ptr(x), ptr_as<float>(w), T, H, E, dtype_code(x), ptr_as<float>(logits), stream_of(x)), "mts_router_wide_fwd");
    else
        check(mts_router_logits_fwd(ptr(x), ptr_as<float>(w), T, H, E, dtype_code(x), ptr_as<float>(logits), stream_of(x)), "mts_router_logits_fwd");
}

void router_projection_backward(const Tensor& g, const Tensor& x, const Tensor& w, const Tensor& dx, const Tensor& dw) {
    const int64_t T = x.size(0), H = x.size(1), E = w.size(0);
    const bool wide = E > kFewExperts;
    const int64_t ws_bytes = wide ? mts_router_wide_bwd_workspace_bytes(T, H, E) : mts_router_logits_bwd_workspace_bytes(T, H, E);
    Tensor ws = bytes(ws_bytes, x);
    check((wide ? mts_router_wide_bwd : mts_router_logits_bwd)(ptr_as<float>(g), ptr(x), ptr_as<float>(w), T, H, E, dtype_code(x), ptr(dx), ptr_as<float>(dw),
                                                               ptr(ws), ws_bytes, stream_of(x)),
          wide ? "mts_router_wide_bwd" : "mts_router_logits_bwd");
}

void router_gradient(const Tensor& x, RouterTail& t, const Tensor& ds) {   // dS and the router's loss terms -> dx_r, dW_r
    const int64_t T = x.size(0), H = x.size(1), E = t.w_r.size(0), K = t.weights.size(1);
    const bool narrow = x.scalar_type() != at::kFloat;
    t.dx_r = at::empty_like(x);
    t.dw_r = at::empty_like(t.w_r);
    Tensor g_w = narrow ? Tensor() : ds, g_w_act = narrow ? ds : Tensor();
    if (t.kept_reverse.defined() && ds.defined()) {
        g_w = at::empty_like(t.weights);
        g_w_act = Tensor();
        check(mts_moe_capacity_weights_bwd(ptr(ds), ptr_as<float>(t.weights), ptr_as<int32_t>(t.kept_reverse), T, K, t.normalize, dtype_code(ds),
                                           ptr_as<float>(g_w), stream_of(x)),
              "mts_moe_capacity_weights_bwd");
    }
    if (E > kFewExperts) {
        Tensor g_logits = at::empty_like(t.logits);
        check(mts_router_bwd(ptr_as<float>(t.logits), ptr_as<float>(t.weights), ptr_as<int32_t>(t.indices), ptr_as<float>(g_w), ptr(g_w_act),
                             narrow ? dtype_code(x) : 0, ptr_as<float>(t.g_prob_mean), ptr_as<float>(t.g_z_loss), ptr_as<float>(t.g_load_balance),
                             ptr_as<int32_t>(t.counts), T, E, K, t.normalize, ptr_as<float>(g_logits), stream_of(x)),
              "mts_router_bwd");
        router_projection_backward(g_logits, x, t.w_r, t.dx_r, t.dw_r);
        return;
    }
    const int64_t ws_bytes = mts_moe_head_bwd_workspace_bytes(T, H, E);
    Tensor ws = bytes(ws_bytes, x);
    check(mts_moe_head_bwd(ptr(x), ptr_as<float>(t.w_r), ptr_as<float>(t.logits), ptr_as<float>(t.weights), ptr_as<int32_t>(t.indices),
                           ptr_as<int32_t>(t.counts), ptr_as<float>(g_w), ptr(g_w_act), ptr_as<float>(t.g_prob_mean),
                           ptr_as<float>(t.g_z_loss), ptr_as<float>(t.g_load_balance), T, H, E, K, t.normalize, dtype_code(x), ptr(t.dx_r),
                           ptr_as<float>(t.dw_r), ptr(ws), ws_bytes, stream_of(x)),
          "mts_moe_head_bwd");
}

ExpertGrads experts_backward(const Saved& s, Tensor dO, const Needs& need, const Options& opt, RouterTail* tail) {
    const int64_t T = s.x.size(0), H = s.x.size(1), E = s.w1.size(0), I = s.w1.size(1) / 2, TK = s.weights.numel(), K = TK / T;
    const auto dtype = s.x.scalar_type();
    const int act = dtype_code(dtype);
    dO = dO.to(dtype).contiguous();
    const int device = s.x.device().index();
    const hipStream_t main = (hipStream_t)stream_of(s.x);
    const bool overlap = opt.on(OVERLAP);
    auto side = [&](int i) { return overlap ? side_stream(device, i) : main; };
    ExpertGrads g;
    Tensor w1_bwd, w2_bwd, d_pre_act, weighted_act, ds_part, ws1, ws2, schedule, dx_expanded;
    Together temporaries(s.x);
    Forked forked(main);   // behind everything that the side streams touch: joined first

    // The ring kernels (16-bit types, widths of whole 64-wide k-tiles or of at least 256) and the fp32 kernels read the
    // weights in their stored layout; other contracts get transposed copies, W1's made on a side stream next to the dO*W2 GEMM.
    const int layout = stored_layout(act, H, I);
    hipStream_t side0 = main;
    if (need.x) {
        if (layout) w1_bwd = s.staged1.defined() ? s.staged1 : stage(s.w1, false, dtype, main);
        else {
            side0 = side(0);
            forked.fork(side0);
            w1_bwd = stage(s.w1, true, dtype, side0);
        }
    }
    w2_bwd = layout && s.staged2.defined() ? s.staged2 : stage(s.w2, !layout, dtype, main);

    const bool weighted = s.post_act.defined();
    weighted_act = weighted ? s.post_act : at::empty({TK, I}, s.x.options());   // s * silu(g) * u
    // When every gradient is wanted, dW1, dW2, dX and the dS reduction go out as ONE launch whose block order starts the long
    // weight-gradient tiles first; which XCD runs which of its units and dX tiles follows a table that the dO * W2 launch
    // writes on the side (uneven routing).
    const bool joint_f32 = opt.on(JOINT_BWD) && need.x && need.w1 && need.w2 && need.s && dtype == at::kFloat && s.w1.scalar_type() == at::kFloat &&
                           s.w2.scalar_type() == at::kFloat && mts_moe_bwd_joint_f32_supported(H, I) && aligned16(dO) && aligned16(s.x) && aligned16(w1_bwd);
    const bool joint = opt.on(JOINT_BWD) && need.x && need.w1 && need.w2 && need.s && layout && s.w1.scalar_type() == s.w2.scalar_type() &&
                       mts_moe_bwd_joint_supported(act, H, I);
    auto dw_workspace = [&](int which, bool wanted) {
        const int64_t n = wanted && dtype != at::kFloat ? mts_moe_bwd_dw_workspace_bytes(which, E, H, I) : 0;
        return n > 0 && n <= opt.dw_workspace_limit ? at::empty({n}, s.x.options().dtype(at::kByte)) : Tensor();
    };
    ws1 = dw_workspace(1, need.w1);
    ws2 = dw_workspace(2, need.w2);
    const int64_t ws1_bytes = ws1.defined() ? ws1.numel() : 0, ws2_bytes = ws2.defined() ? ws2.numel() : 0;
    if (joint && opt.on(JOINT_SCHEDULE) && ws1.defined() && ws2.defined() && mts_moe_bwd_schedule_bytes(E) > 0)
        temporaries.add(schedule, mts_moe_bwd_schedule_bytes(E) / 4, at::kInt);
    temporaries.add(d_pre_act, TK, 2 * I, dtype);
    temporaries.add(ds_part, TK, mts_moe_ds_partials(I), at::kFloat);
    if (need.x) temporaries.add(dx_expanded, TK, H, dtype);
    // the router's backward rides in the joint launch: it needs nothing the launch writes
    const bool tail_in_joint = joint && tail && opt.on(TAIL_IN_JOINT) && mts_moe_bwd_joint_router_supported(act, T, H, I, E);
    const int64_t tail_bytes = tail_in_joint ? mts_moe_head_bwd_workspace_bytes(T, H, E) : 0;
    Tensor tail_ws;
    if (tail_in_joint) {
        temporaries.add(g.ds, T, K, s.weights.scalar_type());
        temporaries.add(tail->dx_r, T, H, dtype);
        temporaries.add(tail_ws, std::max<int64_t>(tail_bytes, 4), at::kByte);
    }
    temporaries.make();
    check(mts_moe_bwd_dy1(ptr(dO), ptr(w2_bwd), layout, ptr(s.pre_act), ptr(s.weights), ptr_as<int32_t>(s.x_gather), ptr_as<int32_t>(s.s_scatter),
                          ptr_as<int32_t>(s.expert_start), T, K, E, H, I, act, ptr(d_pre_act), weighted ? nullptr : ptr(weighted_act),
                          ptr_as<float>(ds_part), ptr_as<int32_t>(schedule), main),
          "mts_moe_bwd_dy1");

    auto combine_dx = [&]() {
        if (tail && !tail->dx_r.defined()) router_gradient(s.x, *tail, g.ds);
        g.dx = at::empty({T, H}, s.x.options());
        check(mts_moe_combine(ptr(dx_expanded), nullptr, tail ? ptr(tail->dx_r) : nullptr, ptr_as<int32_t>(s.s_reverse), T, K, H, act, ptr(g.dx), main),
              "mts_moe_combine");
    };

    if (joint) {
        g.dw1 = at::empty_like(s.w1);
        g.dw2 = at::empty_like(s.w2);
        if (!g.ds.defined()) g.ds = at::empty({T, K}, s.weights.options());
        const int grad = dtype_code(s.w1);
        if (tail_in_joint) {
            tail->dw_r = at::empty_like(tail->w_r);
            if (opt.on(COMBINE_IN_TAIL)) g.dx = at::empty_like(s.x);
            check(mts_moe_bwd_joint_router(ptr(dO), ptr(weighted_act), ptr(d_pre_act), ptr(s.x), ptr(w1_bwd), ptr_as<int32_t>(s.x_gather),
                                           ptr_as<int32_t>(s.expert_start), ptr_as<int32_t>(s.s_reverse), ptr_as<float>(ds_part), T, K, E, H, I, act, grad,
                                           ptr(dx_expanded), ptr(g.dw1), ptr(g.dw2), ptr(g.ds), ptr(ws1), ws1_bytes, ptr(ws2), ws2_bytes,
                                           ptr_as<float>(tail->w_r), ptr_as<float>(tail->logits), ptr_as<float>(tail->weights),
                                           ptr_as<int32_t>(tail->indices), ptr_as<int32_t>(tail->counts), ptr_as<float>(tail->g_prob_mean),
                                           ptr_as<float>(tail->g_z_loss), ptr_as<float>(tail->g_load_balance),
                                           (tail->normalize ? 1 : 0) | (tail->kept_reverse.defined() ? MTS_NORMALIZE_KEPT : 0), ptr(tail->dx_r), ptr(g.dx),
                                           ptr_as<float>(tail->dw_r), ptr(tail_ws), tail_bytes, ptr_as<int32_t>(schedule), main),
                  "mts_moe_bwd_joint_router");
            if (!g.dx.defined()) combine_dx();
            return g;
        }
        check(mts_moe_bwd_joint(ptr(dO), ptr(weighted_act), ptr(d_pre_act), ptr(s.x), ptr(w1_bwd), ptr_as<int32_t>(s.x_gather),
                                ptr_as<int32_t>(s.expert_start), ptr_as<int32_t>(s.s_reverse), ptr_as<float>(ds_part), T, K, E, H, I, act, grad,
                                ptr(dx_expanded), ptr(g.dw1), ptr(g.dw2), ptr(g.ds), ptr(ws1), ws1_bytes, ptr(ws2), ws2_bytes, ptr_as<int32_t>(schedule), main),
              "mts_moe_bwd_joint");
        combine_dx();
        return g;
    }

    if (joint_f32) {
        g.dw1 = at::empty_like(s.w1);
        g.dw2 = at::empty_like(s.w2);
        g.ds = at::empty({T, K}, s.weights.options());
        check(mts_moe_bwd_joint_f32(ptr_as<float>(dO), ptr_as<float>(weighted_act), ptr_as<float>(d_pre_act), ptr_as<float>(s.x), ptr_as<float>(w1_bwd),
                                    ptr_as<int32_t>(s.x_gather), ptr_as<int32_t>(s.expert_start), ptr_as<int32_t>(s.s_reverse), ptr_as<float>(ds_part), T, K, E, H, I,
                                    ptr_as<float>(dx_expanded), ptr_as<float>(g.dw1), ptr_as<float>(g.dw2), ptr_as<float>(g.ds), main),
              "mts_moe_bwd_joint_f32");
        combine_dx();
        return g;
    }

    // dW2, dW1 and dX side by side: the two weight-gradient GEMMs have fewer tiles than the chip has CUs
    const hipStream_t s0 = need.w2 ? side(0) : main, s1 = need.w1 ? side(1) : main;
    if (need.w2) forked.fork(s0);
    if (need.w1) forked.fork(s1);
    // The routing-weight gradient is needed after the join only: it leads one of the side streams (when there is one) so that
    // dX follows the dO*W2 GEMM directly on the caller's stream; the router's gradient wants it on the caller's stream.
    if (need.s) {
        g.ds = at::empty({T, K}, s.weights.options());
        check(mts_moe_bwd_ds(ptr_as<float>(ds_part), ptr_as<int32_t>(s.s_reverse), TK, I, act, ptr(g.ds), tail ? main : (need.w2 ? s0 : s1)), "mts_moe_bwd_ds");
    }
    if (need.w2) {
        g.dw2 = at::empty_like(s.w2);
        check(mts_moe_bwd_dw2(ptr(dO), ptr(weighted_act), ptr_as<int32_t>(s.x_gather), ptr_as<int32_t>(s.expert_start), T, K, E, H, I, act,
                              dtype_code(s.w2), ptr(g.dw2), ptr(ws2), ws2_bytes, s0),
              "mts_moe_bwd_dw2");
    }
    if (need.w1) {
        g.dw1 = at::empty_like(s.w1);
        check(mts_moe_bwd_dw1(ptr(d_pre_act), ptr(s.x), ptr_as<int32_t>(s.x_gather), ptr_as<int32_t>(s.expert_start), T, K, E, H, I, act,
                              dtype_code(s.w1), ptr(g.dw1), ptr(ws1), ws1_bytes, s1),
              "mts_moe_bwd_dw1");
    }
    if (need.x) {
        if (!layout) order_after(main, side0);   // W1's transposed copy
        check(mts_moe_bwd_dx(ptr(d_pre_act), ptr(w1_bwd), layout, ptr_as<int32_t>(s.expert_start), TK, E, H, I, act, ptr(dx_expanded), main), "mts_moe_bwd_dx");
        combine_dx();
    }
    forked.join();
    return g;
}

// ---- autograd nodes ------------------------------------------------------------------------------------------------------------

struct FusedMoE : torch::autograd::Function<FusedMoE> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w1_, const Tensor& w2_, const Tensor& index_, const Tensor& weights_,
                          int64_t switches, int64_t limit) {
        const Options opt{switches, limit};
        const Tensor x = x_.contiguous(), w1 = w1_.contiguous(), w2 = w2_.contiguous(), index = index_.contiguous();
        Saved s;
        Tensor out = experts_forward(x, w1, w2, weights_.contiguous().view(-1), route(index, w1.size(0)), opt, s);
        variable_list keep;
        s.append_to(keep);
        ctx->save_for_backward(std::move(keep));
        ctx->saved_data["options"] = std::vector<int64_t>{switches, limit};
        ctx->set_materialize_grads(false);
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        variable_list result(7);
        if (!grads[0].defined()) return result;
        const auto opt = ctx->saved_data["options"].toIntVector();
        const Saved s(ctx->get_saved_variables());
        c10::OptionalDeviceGuard guard(s.x.device());
        const ExpertGrads g = experts_backward(s, grads[0], {ctx->needs_input_grad(0), ctx->needs_input_grad(1), ctx->needs_input_grad(2), ctx->needs_input_grad(4)},
                                               {opt[0], opt[1]}, nullptr);
        result[0] = g.dx, result[1] = g.dw1, result[2] = g.dw2, result[4] = g.ds;
        return result;
    }
};

// The whole MoE layer (router projection, post-process, routing metadata, experts, combine) as one node.
struct LayerForward {
    Tensor out, load_balance, z_loss, prob_mean, entropy, counts, load_stats, indices, weights;   // results
    Tensor w_r, logits;
    Saved s;
};

// capacity >= 0: an expert accepts at most that many routes; the others get no row
LayerForward layer_forward(const Tensor& x_, const Tensor& w_r_, const Tensor& w1_, const Tensor& w2_, int64_t K, bool normalize, int64_t capacity,
                           const Options& opt) {
    LayerForward f;
    const Tensor x = dense_router_operand(x_, w_r_.size(0)), w_r = dense_router_operand(w_r_, w_r_.size(0));
    const Tensor w1 = w1_.contiguous(), w2 = w2_.contiguous();
    const int64_t T = x.size(0), H = x.size(1), E = w_r.size(0), TK = T * K, I = w1.size(1) / 2;
    const auto dtype = x.scalar_type();
    const bool narrow = dtype != at::kFloat, limited = capacity >= 0, alone = opt.on(NO_BACKWARD), few = E <= kFewExperts;
    // few tokens: all of it behind one entry point, in two launches
    const bool whole = narrow && !limited && opt.on(WEIGHTED_POST) &&
                       mts_moe_few_tokens_preferred(dtype_code(dtype), reads_masters(x, w1, w2, TK, opt) ? MTS_F32 : dtype_code(dtype), T, K, E, H, I);
    const bool chained = few || mts_moe_wide_head_supported(T, H, E, K);   // projection, post-process and routing metadata behind one entry point
    const int64_t ws_bytes = whole ? (H + 31) / 32 * 4 : few ? mts_moe_head_workspace_bytes(T, K, E) : chained ? mts_moe_wide_head_workspace_bytes(T, E) : mts_moe_router_route_workspace_bytes(T, K, E);
    f.w_r = w_r;
    f.weights = f32({T, K}, x);
    // The integer results in one allocation and the fp32 statistics in another: a caller may save all results together, which torch refuses
    // for one storage under two types.
    const int64_t counts_bytes = (E + 3) / 4 * 16;
    const Tensor integers = i32({counts_bytes / 4 + TK}, x);
    f.counts = part_of(integers, 0, {E}, at::kInt), f.indices = part_of(integers, counts_bytes, {T, K}, at::kInt);
    Tensor weights_act, ws, post_act, y;
    Routing r;
    // what the backward pass keeps, and what this call alone needs
    Together kept(x), scratch(x);
    Together& own = alone ? scratch : kept;
    own.add(f.logits, T, E, at::kFloat);
    if (narrow || limited) own.add(weights_act, T, K, dtype);
    else weights_act = f.weights;
    auto add_rows = [&](Routing& to) {
        own.add(to.expert_start, E + 1, at::kInt);
        own.add(to.s_scatter, TK, at::kInt);
        own.add(to.s_reverse, TK, at::kInt);
        own.add(to.x_gather, TK, at::kInt);
    };
    add_rows(r);
    scratch.add(ws, std::max<int64_t>(ws_bytes, 4), at::kByte);
    scratch.add(y, TK, H, dtype);
    if (alone) scratch.add(post_act, TK, I, dtype);
    scratch.make();
    if (!alone) kept.make();
    // E mean probabilities, z, entropy, load-balancing term, E + 7 load statistics
    Tensor stats = f32({2 * E + 10}, x);
    if (alone) {   // nobody differentiates: parts instead of views
        auto floats_at = [&](int64_t first, at::IntArrayRef size) { return part_of(stats, first * 4, size, at::kFloat); };
        f.prob_mean = floats_at(0, {E}), f.z_loss = floats_at(E, {}), f.entropy = floats_at(E + 1, {}), f.load_balance = floats_at(E + 2, {});
        f.load_stats = floats_at(E + 3, {E + 7});
    } else {
        f.prob_mean = stats.narrow(0, 0, E), f.z_loss = stats.select(0, E), f.entropy = stats.select(0, E + 1), f.load_balance = stats.select(0, E + 2);
        f.load_stats = stats.narrow(0, E + 3, E + 7);
    }
    void* load_stats = limited ? nullptr : ptr(f.load_stats);
    void* cast_weights = narrow && !limited ? ptr(weights_act) : nullptr;
    if (whole) {
        const auto [w1_read, w2_read] = forward_weights(x, w1, w2, TK, opt);
        Tensor pre_act;
        if (!alone) pre_act = at::empty({TK, 2 * I}, x.options()), post_act = at::empty({TK, I}, x.options());
        f.out = at::empty({T, H}, x.options());
        check(mts_moe_few_tokens_fwd(ptr(x), ptr_as<float>(w_r), ptr(w1_read), ptr(w2_read), dtype_code(w1_read), T, H, E, I, K, normalize, dtype_code(dtype),
                                     ptr_as<float>(f.logits), ptr_as<float>(f.weights), ptr_as<int32_t>(f.indices), cast_weights, ptr_as<float>(f.prob_mean),
                                     ptr_as<float>(f.z_loss), ptr_as<float>(f.entropy), ptr_as<int32_t>(f.counts), ptr_as<float>(f.load_balance),
                                     static_cast<float*>(load_stats), ptr_as<int32_t>(r.expert_start), ptr_as<int32_t>(r.s_scatter), ptr_as<int32_t>(r.s_reverse),
                                     ptr_as<int32_t>(r.x_gather), ptr(pre_act), ptr(post_act), ptr(y), ptr_as<int32_t>(ws), ptr(f.out), stream_of(x)),
              "mts_moe_few_tokens_fwd");
        keep(f.s, x, w1, w2, w1_read, w2_read, pre_act, post_act, weights_act, r);
        return f;
    }
    Tensor copy1, copy2;   // of master weights: made beside the head
    if (chained) {
        MtsCast casts[2];
        const bool ride = copies_masters(x, w1, w2) && mts_moe_head_casts_ride(T, H, E, dtype_code(x), w1.numel(), w2.numel());
        const bool copied = copies_masters(x, w1, w2) && !reads_masters(x, w1, w2, TK, opt, ride);
        if (copied) {
            copy1 = at::empty(w1.sizes(), x.options()), copy2 = at::empty(w2.sizes(), x.options());
            casts[0] = {ptr_as<float>(w1), ptr(copy1), w1.numel()}, casts[1] = {ptr_as<float>(w2), ptr(copy2), w2.numel()};
        }
        check((few ? mts_moe_head_cast_fwd : mts_moe_wide_head_cast_fwd)(ptr(x), ptr_as<float>(w_r), T, H, E, K, normalize, dtype_code(x), ptr_as<float>(f.logits), ptr_as<float>(f.weights),
                               ptr_as<int32_t>(f.indices), cast_weights, ptr_as<float>(f.prob_mean), ptr_as<float>(f.z_loss), ptr_as<float>(f.entropy),
                               ptr_as<int32_t>(f.counts), ptr_as<float>(f.load_balance), static_cast<float*>(load_stats), ptr_as<int32_t>(r.expert_start),
                               ptr_as<int32_t>(r.s_scatter), ptr_as<int32_t>(r.s_reverse), ptr_as<int32_t>(r.x_gather), ptr(ws), ws_bytes,
                               copied ? casts : nullptr, stream_of(x)),
              few ? "mts_moe_head_cast_fwd" : "mts_moe_wide_head_cast_fwd");
    } else {
        router_projection_forward(x, w_r, f.logits);
        check(mts_moe_router_route(ptr_as<float>(f.logits), T, E, K, normalize, ptr_as<float>(f.weights), ptr_as<int32_t>(f.indices), ptr_as<float>(f.prob_mean),
                                   ptr_as<float>(f.z_loss), ptr_as<float>(f.entropy), ptr_as<int32_t>(f.counts), ptr_as<float>(f.load_balance),
                                   static_cast<float*>(load_stats), cast_weights, narrow ? dtype_code(x) : 0, ptr_as<int32_t>(r.expert_start),
                                   ptr_as<int32_t>(r.s_scatter), ptr_as<int32_t>(r.s_reverse), ptr_as<int32_t>(r.x_gather), ptr(ws), ws_bytes, stream_of(x)),
              "mts_moe_router_route");
    }
    if (limited) {
        const Routing every = r;
        Tensor accepted, keys;
        const int64_t keys_bytes = mts_moe_capacity_compact_workspace_bytes(T, K);
        Together rows(x);
        rows.add(r.expert_start, E + 1, at::kInt);
        rows.add(r.s_scatter, TK, at::kInt);
        rows.add(r.s_reverse, TK, at::kInt);
        rows.add(r.x_gather, TK, at::kInt);
        rows.add(accepted, E, at::kInt);
        rows.add(keys, std::max<int64_t>(keys_bytes, 4), at::kByte);
        rows.make();
        check(mts_moe_capacity_compact(ptr_as<float>(f.weights), ptr_as<int32_t>(f.counts), ptr_as<int32_t>(every.expert_start),
                                       ptr_as<int32_t>(every.s_scatter), T, K, E, capacity, ptr_as<int32_t>(accepted), ptr_as<int32_t>(r.expert_start),
                                       ptr_as<int32_t>(r.s_scatter), ptr_as<int32_t>(r.s_reverse), ptr_as<int32_t>(r.x_gather), ptr(keys), keys_bytes,
                                       stream_of(x)),
              "mts_moe_capacity_compact");
        check(mts_moe_capacity_weights_fwd(ptr_as<float>(f.weights), ptr_as<int32_t>(r.s_reverse), ptr_as<int32_t>(accepted), ptr_as<float>(f.entropy), T, K,
                                           E, normalize, dtype_code(x), ptr(weights_act), ptr_as<float>(f.load_stats), stream_of(x)),
              "mts_moe_capacity_weights_fwd");
    }
    f.out = experts_forward(x, w1, w2, weights_act, r, opt, f.s, post_act, y, copy1, copy2);
    return f;
}

struct MoELayer : torch::autograd::Function<MoELayer> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& w_r, const Tensor& w1, const Tensor& w2, int64_t K, bool normalize,
                                 int64_t capacity, int64_t switches, int64_t limit) {
        const LayerForward f = layer_forward(x, w_r, w1, w2, K, normalize, capacity, {switches, limit});
        variable_list keep;
        f.s.append_to(keep);
        keep.insert(keep.end(), {f.w_r, f.logits, f.weights, f.indices, f.counts});
        ctx->save_for_backward(std::move(keep));
        ctx->saved_data["options"] = std::vector<int64_t>{switches, limit, normalize, capacity >= 0};
        ctx->mark_non_differentiable({f.entropy, f.counts, f.load_stats, f.indices, f.weights});
        ctx->set_materialize_grads(false);
        return {f.out, f.load_balance, f.z_loss, f.prob_mean, f.entropy, f.counts, f.load_stats, f.indices, f.weights};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto o = ctx->saved_data["options"].toIntVector();
        const variable_list saved = ctx->get_saved_variables();
        const Saved s(saved);
        const Tensor* router = &saved[Saved::kCount];
        c10::OptionalDeviceGuard guard(s.x.device());
        RouterTail tail{router[0], router[1], router[2], router[3], router[4], like_f32(grads[3]), like_f32(grads[2]), like_f32(grads[1]), o[2] != 0,
                        o[3] ? s.s_reverse : Tensor(), {}, {}};
        const bool need_x = ctx->needs_input_grad(0), need_wr = ctx->needs_input_grad(1);
        const bool wants_router = need_x || need_wr;
        variable_list result(9);
        if (grads[0].defined()) {
            const ExpertGrads g = experts_backward(s, grads[0], {need_x, ctx->needs_input_grad(2), ctx->needs_input_grad(3), wants_router}, {o[0], o[1]},
                                                   wants_router ? &tail : nullptr);
            if (wants_router && !tail.dw_r.defined()) router_gradient(s.x, tail, g.ds);   // x needs no gradient: no dX combine
            result[0] = g.dx, result[2] = g.dw1, result[3] = g.dw2;
        } else if (wants_router) {   // only the router's loss terms reach this layer
            router_gradient(s.x, tail, Tensor());
            if (need_x) result[0] = tail.dx_r;
        }
        if (need_wr) result[1] = tail.dw_r;
        return result;
    }
};

struct RouterPostprocess : torch::autograd::Function<RouterPostprocess> {
    static variable_list forward(AutogradContext* ctx, const Tensor& logits_, int64_t K, bool normalize, int64_t act_dtype) {
        const Tensor logits = logits_.contiguous();
        const int64_t T = logits.size(0), E = logits.size(1);
        const bool cast = act_dtype >= 0;
        Tensor weights = f32({T, K}, logits), indices = i32({T, K}, logits), counts = i32({E}, logits);
        Tensor stats = f32({2 * E + 10}, logits);   // E + 3 statistics, E + 7 load statistics
        Tensor prob_mean = stats.narrow(0, 0, E), z_loss = stats.select(0, E), entropy = stats.select(0, E + 1), load_balance = stats.select(0, E + 2),
               load_stats = stats.narrow(0, E + 3, E + 7);
        // the copy of the weights in the activation dtype, written by the same kernel (what the router module otherwise makes
        // with tensor.to(): one launch forward, one backward)
        Tensor weights_act;
        if (cast) weights_act = at::empty({T, K}, logits.options().dtype(act_dtype == MTS_BF16 ? at::kBFloat16 : at::kHalf));
        const int64_t ws_bytes = mts_router_workspace_bytes(T, E);
        Tensor ws = bytes(ws_bytes, logits);
        check(mts_router_fwd(ptr_as<float>(logits), T, E, K, normalize, ptr_as<float>(weights), ptr_as<int32_t>(indices), ptr_as<float>(prob_mean),
                             ptr_as<float>(z_loss), ptr_as<float>(entropy), ptr_as<int32_t>(counts), ptr_as<float>(load_balance), ptr_as<float>(load_stats),
                             ptr(weights_act), cast ? (int)act_dtype : 0, ptr(ws), ws_bytes, stream_of(logits)),
              "mts_router_fwd");
        ctx->save_for_backward({logits, weights, indices, counts});
        ctx->saved_data["options"] = std::vector<int64_t>{K, normalize, cast ? act_dtype : 0};
        ctx->mark_non_differentiable({indices, entropy, counts, load_stats});
        ctx->set_materialize_grads(false);   // no zero tensors for the outputs that took no part in the loss
        variable_list out{weights, indices, prob_mean, z_loss, entropy, counts, load_balance, load_stats};
        if (cast) out.push_back(weights_act);
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const auto o = ctx->saved_data["options"].toIntVector();
        c10::OptionalDeviceGuard guard(s[0].device());
        const Tensor g_w = like_f32(grads[0]), g_p = like_f32(grads[2]), g_z = like_f32(grads[3]), g_lb = like_f32(grads[6]);
        const Tensor g_act = grads.size() > 8 && grads[8].defined() ? grads[8].contiguous() : Tensor();   // stays in the activation dtype
        Tensor g_logits = at::empty_like(s[0]);
        check(mts_router_bwd(ptr_as<float>(s[0]), ptr_as<float>(s[1]), ptr_as<int32_t>(s[2]), ptr_as<float>(g_w), ptr(g_act), (int)o[2], ptr_as<float>(g_p),
                             ptr_as<float>(g_z), ptr_as<float>(g_lb), ptr_as<int32_t>(s[3]), s[0].size(0), s[0].size(1), o[0], o[1], ptr_as<float>(g_logits),
                             stream_of(s[0])),
              "mts_router_bwd");
        return {g_logits, Tensor(), Tensor(), Tensor()};
    }
};

// logits = float(x) @ W_r^T without the fp32 copy of x; backward gives dx in x's dtype.
struct RouterLogits : torch::autograd::Function<RouterLogits> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {   // dense
        Tensor logits = f32({x.size(0), w.size(0)}, x);
        router_projection_forward(x, w, logits);
        ctx->save_for_backward({x, w});
        return logits;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        c10::OptionalDeviceGuard guard(s[0].device());
        if (written_out(grads)) {
            const Tensor wide = grads[0].to(at::kFloat);
            return {wide.matmul(s[1]).to(s[0].scalar_type()), wide.t().matmul(s[0].to(at::kFloat))};
        }
        const Tensor g = dense_router_operand(grads[0].to(at::kFloat), s[1].size(0));
        Tensor dx = at::empty_like(s[0]), dw = at::empty_like(s[1]);
        router_projection_backward(g, s[0], s[1], dx, dw);
        return {dx, dw};
    }
};

// ---- the decoder's dense operators -----------------------------------------------------------------------------------------------

// Each gives way to stock operators where all_plain() does not hold, and computes its gradients with them where
// written_out() says so.

bool rmsnorm_supported(const Tensor& x, const Tensor& w, const MaybeTensor& residual) {
    if (!(all_plain(x, w) && (!residual || is_plain(*residual)) && on_one_gpu(x, w) && is_activation_type(x.scalar_type()) &&
          w.scalar_type() == at::kFloat && w.dim() == 1 && x.dim() >= 1 && x.size(-1) == w.size(0) && x.numel() > 0 && x.numel() / x.size(-1) < MTS_MAX_NORM_ROWS && mts_rmsnorm_supported(x.size(-1))))
        return false;
    return !residual || (on_one_gpu(x, *residual) && residual->scalar_type() == x.scalar_type() && residual->sizes() == x.sizes());
}

// y, or (x + residual, y) with a residual
struct RMSNorm : torch::autograd::Function<RMSNorm> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const MaybeTensor& residual_, const Tensor& w, double eps) {   // dense16
        const int64_t H = x.size(-1), N = x.numel() / H;
        Tensor residual, total = x, y = at::empty_like(x), rstd = f32({N}, x);
        if (residual_) {
            residual = *residual_;
            total = at::empty_like(x);
        }
        check(mts_rmsnorm_fwd(ptr(x), ptr(residual), ptr_as<float>(w), N, H, eps, dtype_code(x), residual_ ? ptr(total) : nullptr, ptr(y), ptr_as<float>(rstd),
                              stream_of(x)),
              "mts_rmsnorm_fwd");
        ctx->save_for_backward({total, w, rstd});
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        if (residual_) return {total, y};
        return {y};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const bool with_sum = grads.size() == 2;
        Tensor g_sum = with_sum ? grads[0] : Tensor(), g_y = grads.back();
        if (!g_y.defined()) return {g_sum, with_sum ? g_sum : Tensor(), Tensor(), Tensor()};   // only the residual stream goes on
        c10::OptionalDeviceGuard guard(s[0].device());
        const int64_t H = s[0].size(-1), N = s[0].numel() / H, ws_bytes = mts_rmsnorm_bwd_workspace_bytes(N, H);
        if (written_out(grads)) {
            const Tensor v = s[0].to(at::kFloat), r = at::rsqrt(v.square().mean(-1, true) + ctx->saved_data["eps"].toDouble()), n = v * r;
            const Tensor gy = g_y.to(at::kFloat), gw = gy * s[1];
            Tensor d = r * (gw - n * (gw * n).mean(-1, true));
            if (g_sum.defined()) d = d + g_sum.to(at::kFloat);
            d = d.to(s[0].scalar_type());
            return {d, with_sum ? d : Tensor(), (gy * n).reshape({N, H}).sum(0), Tensor()};
        }
        g_y = dense16(g_y);
        if (g_sum.defined()) g_sum = dense16(g_sum);
        Tensor d_sum = at::empty_like(s[0]), dw = at::empty_like(s[1]), ws = bytes(ws_bytes, s[0]);
        check(mts_rmsnorm_bwd(ptr(g_y), ptr(g_sum), ptr(s[0]), ptr_as<float>(s[1]), ptr_as<float>(s[2]), N, H, dtype_code(s[0]), ptr(d_sum), ptr_as<float>(dw),
                              ptr(ws), ws_bytes, stream_of(s[0])),
              "mts_rmsnorm_bwd");
        return {d_sum, with_sum ? d_sum : Tensor(), dw, Tensor()};
    }
};

enum RopeMode : int64_t { TURN = 0, TURN_BACK = 1, COPY = 2 };

bool rope_table_fits(const Tensor& t, const Tensor& like, int64_t S, int64_t D) {
    return on_one_gpu(like, t) && t.scalar_type() == like.scalar_type() && t.dim() == 2 && t.size(0) == S && t.size(1) == D && t.is_contiguous() && !t.requires_grad();
}
bool rope_supported(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin) {
    if (!(all_plain(q, k, cos, sin) && on_one_gpu(q, k) && q.dim() == 4 && q.sizes() == k.sizes() && q.scalar_type() == k.scalar_type() &&
          is_activation_type(q.scalar_type()) && q.numel() > 0))
        return false;
    const int64_t S = q.size(2), D = q.size(3);
    return D % 2 == 0 && q.numel() / 2 < MTS_MAX_ROPE_PAIRS && rope_table_fits(cos, q, S, D) && rope_table_fits(sin, q, S, D);
}
bool qkv_rope_supported(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t heads) {
    if (!(all_plain(qkv, cos, sin) && qkv.is_cuda() && qkv.dim() == 3 && is_activation_type(qkv.scalar_type()) && qkv.numel() > 0 && qkv.size(2) % (3 * heads) == 0)) return false;
    const int64_t S = qkv.size(1), D = qkv.size(2) / (3 * heads);
    return D % 2 == 0 && qkv.numel() / 6 < MTS_MAX_ROPE_PAIRS && rope_table_fits(cos, qkv, S, D) && rope_table_fits(sin, qkv, S, D);
}

struct RopeJob {
    Tensor in, out;   // [B, heads, S, D], any strides but a dense last dimension
    int64_t mode;
};
void launch_rope(const std::vector<RopeJob>& jobs, const Tensor& cos, const Tensor& sin) {
    MtsRopeTensor array[3];
    for (size_t i = 0; i < jobs.size(); ++i) {
        const Tensor &a = jobs[i].in, &b = jobs[i].out;
        array[i] = {ptr(a), ptr(b), a.stride(0), a.stride(2), a.stride(1), b.stride(0), b.stride(2), b.stride(1), (int)jobs[i].mode};
    }
    const Tensor& t = jobs[0].in;
    check(mts_rope(array, (int)jobs.size(), ptr(cos), ptr(sin), t.size(0), t.size(2), t.size(1), t.size(3), dtype_code(t), stream_of(t)), "mts_rope");
}
Tensor dense_rows(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }
// [B, S, heads, D] in memory, as the projection that queries and keys are views of.  A tensor of its own: autograd lets nobody
// change the view that a node returns.
Tensor heads_inside(const Tensor& like, int64_t B, int64_t heads, int64_t S, int64_t D) {
    return at::empty_strided({B, heads, S, D}, {S * heads * D, D, heads * D, 1}, like.options());
}

// the gradient of a turn in stock operators: the pairs turned back
Tensor turned_back(const Tensor& g, const Tensor& cos, const Tensor& sin) {
    const variable_list h = (g * sin).chunk(2, -1);
    return g * cos + at::cat({h[1], -h[0]}, -1);
}

struct Rope : torch::autograd::Function<Rope> {
    static variable_list turn(const Tensor& q_, const Tensor& k_, const Tensor& cos, const Tensor& sin, int64_t mode) {
        const Tensor q = dense_rows(q_), k = dense_rows(k_);
        Tensor a = heads_inside(q, q.size(0), q.size(1), q.size(2), q.size(3)), b = heads_inside(q, q.size(0), q.size(1), q.size(2), q.size(3));
        launch_rope({{q, a, mode}, {k, b, mode}}, cos, sin);
        return {a, b};
    }
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin) {
        ctx->save_for_backward({cos, sin});
        return turn(q, k, cos, sin, TURN);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        c10::OptionalDeviceGuard guard(s[0].device());
        if (written_out(grads)) return {turned_back(grads[0], s[0], s[1]), turned_back(grads[1], s[0], s[1]), Tensor(), Tensor()};
        const variable_list g = turn(grads[0], grads[1], s[0], s[1], TURN_BACK);
        return {g[0], g[1], Tensor(), Tensor()};
    }
};

// Packed projection [B, S, 3 * heads * D] to rotated queries, rotated keys and values [B, heads, S, D].  The values stay where
// they are; the backward launch writes the gradient of the projection in one piece.
struct QkvRope : torch::autograd::Function<QkvRope> {
    static variable_list forward(AutogradContext* ctx, const Tensor& qkv_, const Tensor& cos, const Tensor& sin, int64_t heads) {
        const Tensor qkv = qkv_.contiguous();
        const int64_t B = qkv.size(0), S = qkv.size(1), D = qkv.size(2) / (3 * heads);
        const Tensor parts = qkv.view({B, S, 3, heads, D});
        Tensor q = heads_inside(qkv, B, heads, S, D), k = heads_inside(qkv, B, heads, S, D);
        launch_rope({{parts.select(2, 0).transpose(1, 2), q, TURN}, {parts.select(2, 1).transpose(1, 2), k, TURN}}, cos, sin);
        ctx->save_for_backward({cos, sin});
        ctx->saved_data["heads"] = heads;
        ctx->set_materialize_grads(false);
        return {q, k, parts.select(2, 2).transpose(1, 2)};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor* first = nullptr;
        int given = 0;
        for (const Tensor& g : grads)
            if (g.defined()) {
                ++given;
                first = &g;
            }
        if (!first) return variable_list(4);
        c10::OptionalDeviceGuard guard(s[0].device());
        const int64_t B = first->size(0), heads = first->size(1), S = first->size(2), D = first->size(3);
        if (written_out(grads)) {
            auto part = [&](int i) { return (!grads[i].defined() ? at::zeros_like(*first) : i < 2 ? turned_back(grads[i], s[0], s[1]) : grads[i]).transpose(1, 2); };
            return {at::stack({part(0), part(1), part(2)}, 2).reshape({B, S, 3 * heads * D}), Tensor(), Tensor(), Tensor()};
        }
        // zeros where a part took no part in the loss
        Tensor out = given == 3 ? at::empty({B, S, 3, heads, D}, first->options()) : at::zeros({B, S, 3, heads, D}, first->options());
        std::vector<RopeJob> jobs;
        for (int i = 0; i < 3; ++i)
            if (grads[i].defined()) jobs.push_back({dense_rows(grads[i]), out.select(2, i).transpose(1, 2), i < 2 ? TURN_BACK : COPY});
        launch_rope(jobs, s[0], s[1]);
        return {out.view({B, S, 3 * heads * D}), Tensor(), Tensor(), Tensor()};
    }
};

// The projection on a vocabulary: both gradients are this framework's, over whole rounds of tiles (mts_linear_dx_rounds).  They are ahead
// of the library's from 128 rows on (768 wide, us, dX and dW, here / library: 24 576 rows of 50 257 1610 / 2577 and 1520 / 2199, 4096 rows
// 279 / 555 and 278 / 375, 512 rows 69 / 197 and 58 / 67; 1024 rows of 8192 31 / 44 and 26 / 25), and dX no longer where a projection
// is less than eight times as wide as its input (12 288 rows of 2304 48 / 45, 8192 rows of 4096 -> 12 288 612 / 594).
constexpr int64_t kLinearRoundsRows = 128;
int64_t row_pitch(int64_t N) { return (N + 63) / 64 * 64; }   // 16-bit rows that start on 128 bytes
bool linear_in_rounds(const Tensor& x, int64_t T, int64_t N, int64_t K) {
    return T >= kLinearRoundsRows && N >= 8 * K && N < k2GiB && mts_linear_rounds_supported(dtype_code(x), T, N, K, row_pitch(N));
}
// Rows that mts_linear_dx_rounds and mts_linear_dw_rounds read in place, in whole pieces of eight elements: the storage holds the last one too.
bool rows_fit(const Tensor& g) {
    const int64_t end = g.storage_offset() + (g.size(0) - 1) * g.stride(0) + (g.size(1) + 7) / 8 * 8;
    return g.stride(1) == 1 && g.stride(0) >= g.size(1) && g.stride(0) % 8 == 0 && aligned16(g) && end * g.element_size() <= (int64_t)g.storage().nbytes();
}

// Operands of a projection under autocast.
bool projection_operands(const Tensor& x, const Tensor& w) {
    return all_plain(x, w) && on_one_gpu(x, w) && x.dim() >= 2 && w.dim() == 2 && w.scalar_type() == at::kFloat &&
           (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kHalf) && x.size(-1) == w.size(1) && x.numel() > 0 &&
           at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) == x.scalar_type();
}
// The product, where its kernel is ahead of the library's and takes the activations as they lie; else undefined.
Tensor own_product(const Tensor& x, const Tensor& rounded) {
    const int64_t N = rounded.size(0), K = rounded.size(1), T = x.numel() / K;
    if (!mts_linear_fwd_preferred(dtype_code(x), T, N, K) || !x.is_contiguous() || !aligned16(x)) return {};
    const Tensor w = dense16(rounded);
    c10::SmallVector<int64_t, 4> size(x.sizes());
    size.back() = N;
    Tensor y = at::empty(size, x.options());
    check(mts_linear_fwd(ptr(x), ptr(w), T, N, K, dtype_code(x), ptr(y), stream_of(x)), "mts_linear_fwd");
    return y;
}

// A projection whose fp32 weight wants a gradient, which is summed in fp32 here; the products are the library's or ours.
bool linear_supported(const Tensor& x, const Tensor& w) {
    if (!(at::GradMode::is_enabled() && w.requires_grad() && projection_operands(x, w))) return false;
    const int64_t T = x.numel() / x.size(-1), N = w.size(0), K = w.size(1);
    return linear_in_rounds(x, T, N, K) || mts_linear_dw_supported(dtype_code(x), T, N, K);
}

// One that wants none: the weight rounded as autocast does it, and kept by it for as long.
bool linear_alone_supported(const Tensor& x, const Tensor& w) {
    if ((at::GradMode::is_enabled() && (x.requires_grad() || w.requires_grad())) || !projection_operands(x, w)) return false;
    return x.is_contiguous() && aligned16(x) && mts_linear_fwd_preferred(dtype_code(x), x.numel() / x.size(-1), w.size(0), w.size(1));
}
Tensor linear_alone(const Tensor& x, const Tensor& w) { return own_product(x, at::autocast::cached_cast(x.scalar_type(), w, c10::DeviceType::CUDA)); }

struct Linear : torch::autograd::Function<Linear> {
    static variable_list in_rounds(AutogradContext* ctx, const Tensor& g, const Tensor& x, const Tensor& rounded, int64_t T, int64_t N, int64_t K) {
        Tensor dx, dw;
        auto workspace = [&](int which, int64_t& size) {
            size = mts_linear_rounds_workspace_bytes(which, T, N, K);
            return size ? bytes(size, x) : Tensor();
        };
        int64_t size = 0;
        if (ctx->needs_input_grad(0)) {
            const Tensor w = dense16(rounded), ws = workspace(0, size);
            dx = at::empty({T, K}, x.options());
            check(mts_linear_dx_rounds(ptr(g), g.stride(0), ptr(w), T, N, K, dtype_code(x), ptr(dx), ptr(ws), size, stream_of(x)), "mts_linear_dx_rounds");
            dx = dx.view(x.sizes());
        }
        if (ctx->needs_input_grad(1)) {
            const Tensor in = dense16(x.reshape({T, K})), ws = workspace(1, size);
            dw = f32({N, K}, x);
            check(mts_linear_dw_rounds(ptr(g), g.stride(0), ptr(in), T, N, K, dtype_code(x), ptr_as<float>(dw), ptr(ws), size, stream_of(x)),
                  "mts_linear_dw_rounds");
        }
        return {dx, dw};
    }
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
        const Tensor rounded = w.to(x.scalar_type());
        ctx->save_for_backward({x, rounded});
        ctx->saved_data["weight"] = w;   // not kept as it is now: the caller may change it before the backward pass, as under stock autocast
        const Tensor own = own_product(x, rounded);
        return own.defined() ? own : at::linear(x, rounded);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &x = s[0], &rounded = s[1];
        c10::OptionalDeviceGuard guard(x.device());
        const int64_t N = rounded.size(0), K = rounded.size(1), T = x.numel() / K;
        const bool rounds = linear_in_rounds(x, T, N, K);
        if (written_out(grads)) {
            const Tensor g = grads[0].reshape({T, N});
            const Tensor now = ctx->saved_data["weight"].toTensor().to(x.scalar_type());   // for its derivative; the value is that of the forward pass
            const Tensor dx = at::matmul(g, rounded + (now - now.detach())).view(x.sizes());
            // an fp32 copy of the gradient of as many logits would be larger than all else: stock autocast's product there
            if (rounds) return {dx, at::matmul(g.t(), x.reshape({T, K})).to(at::kFloat)};
            return {dx, at::matmul(g.to(at::kFloat).t().contiguous(), x.reshape({T, K}).to(at::kFloat))};
        }
        if (rounds) {
            // Rows at odd places are copied.  us, copy and both gradients / the library's products, 50 257 columns, 768 wide: 24 576 rows 3909 / 4712,
            // 8192 1390 / 1375, 2048 403 / 597, 512 180 / 325, 128 116 / 305; 1024 rows of 8193 66 / 76.
            Tensor g = grads[0].reshape({T, N});
            if (!rows_fit(g) || !mts_linear_rounds_supported(dtype_code(x), T, N, K, g.stride(0)))
                g = at::empty({T, row_pitch(N)}, g.options()).narrow(1, 0, N).copy_(g);
            return in_rounds(ctx, g, x, rounded, T, N, K);
        }
        const Tensor g = dense16(grads[0].reshape({T, N})), in = dense16(x.reshape({T, K}));
        Tensor dx, dw;
        if (ctx->needs_input_grad(0)) {
            if (mts_linear_dx_preferred(dtype_code(x), T, N, K)) {
                const Tensor w = dense16(rounded);
                dx = at::empty(x.sizes(), x.options());
                check(mts_linear_dx(ptr(g), ptr(w), T, N, K, dtype_code(x), ptr(dx), stream_of(x)), "mts_linear_dx");
            } else dx = at::matmul(g, rounded).view(x.sizes());
        }
        if (ctx->needs_input_grad(1)) {
            dw = f32({N, K}, x);
            const int64_t ws_bytes = mts_linear_dw_workspace_bytes(T, N, K);
            Tensor ws = ws_bytes ? bytes(ws_bytes, x) : Tensor();
            check(mts_linear_dw(ptr(g), ptr(in), T, N, K, dtype_code(x), ptr_as<float>(dw), ptr(ws), ws_bytes, stream_of(x)), "mts_linear_dw");
        }
        return {dx, dw};
    }
};

// The stock lookup; the table's gradient is summed here, from the gradient as it arrives in the activation dtype.
bool embedding_supported(const Tensor& ids, const Tensor& w, at::ScalarType type) {
    return at::GradMode::is_enabled() && w.requires_grad() && all_plain(ids, w) && on_one_gpu(ids, w) && ids.scalar_type() == at::kLong && w.dim() == 2 &&
           w.scalar_type() == at::kFloat && is_activation_type(type) && mts_embedding_bwd_preferred(ids.numel(), w.size(0), w.size(1));
}

struct Embedding : torch::autograd::Function<Embedding> {
    static Tensor forward(AutogradContext* ctx, const Tensor& ids, const Tensor& w, at::ScalarType type) {
        ctx->save_for_backward({ids});
        ctx->saved_data["rows"] = w.size(0);
        return at::embedding(w, ids).to(type);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const Tensor ids = ctx->get_saved_variables()[0].contiguous();
        c10::OptionalDeviceGuard guard(ids.device());
        const int64_t V = ctx->saved_data["rows"].toInt(), T = ids.numel(), H = grads[0].size(-1);
        if (written_out(grads)) return {Tensor(), at::embedding_dense_backward(grads[0].to(at::kFloat), ids, V, -1, false), Tensor()};
        const Tensor g = dense16(grads[0]);
        const int64_t ws_bytes = mts_embedding_bwd_workspace_bytes(T, V, H);
        Tensor dw = f32({V, H}, g), ws = bytes(ws_bytes, g);
        check(mts_embedding_bwd(ptr(g), ptr_as<int64_t>(ids), T, V, H, dtype_code(g), ptr_as<float>(dw), ptr(ws), ws_bytes, stream_of(g)), "mts_embedding_bwd");
        return {Tensor(), dw, Tensor()};
    }
};

bool heads_fit(const Tensor& t) {   // as the kernels read them
    return t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 && aligned16(t);
}
bool attention_supported(const Tensor& q, const Tensor& k, const Tensor& v) {
    if (!(all_plain(q, k, v) && on_one_gpu(q, k, v) && q.dim() == 4 && k.sizes() == q.sizes() &&
          v.sizes() == q.sizes() && (q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf) && k.scalar_type() == q.scalar_type() &&
          v.scalar_type() == q.scalar_type() && mts_attention_supported(q.size(0), q.size(1), q.size(2), q.size(3))))
        return false;
    // what the caller has chosen for the stock operator stays chosen: another type, another implementation
    if (at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != q.scalar_type()) return false;
    return at::globalContext().userEnabledFlashSDP() && heads_fit(q) && heads_fit(k) && heads_fit(v);
}

struct Attention : torch::autograd::Function<Attention> {
    static MtsHeads view(const Tensor& t) { return {ptr(t), t.stride(0), t.stride(1), t.stride(2)}; }
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, bool causal) {
        const int64_t B = q.size(0), heads = q.size(1), S = q.size(2);
        Tensor out = heads_inside(q, B, heads, S, q.size(3)), lse = f32({B * heads * S}, q);
        const MtsHeads vq = view(q), vk = view(k), vv = view(v), vo = view(out);
        check(mts_attention_fwd(&vq, &vk, &vv, B, heads, S, causal, dtype_code(q), &vo, ptr_as<float>(lse), stream_of(q)), "mts_attention_fwd");
        ctx->save_for_backward({q, k, v, out, lse});
        ctx->saved_data["causal"] = causal;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &q = s[0], &k = s[1], &v = s[2];
        c10::OptionalDeviceGuard guard(q.device());
        const bool causal = ctx->saved_data["causal"].toBool();
        const int64_t B = q.size(0), heads = q.size(1), S = q.size(2), D = q.size(3);
        if (written_out(grads)) {   // in fp32
            const double scale = 1.0 / std::sqrt((double)D);
            const Tensor qf = q.to(at::kFloat), kf = k.to(at::kFloat), vf = v.to(at::kFloat), g = grads[0].to(at::kFloat);
            Tensor score = at::matmul(qf, kf.transpose(2, 3).contiguous()) * scale;
            if (causal) score = score.masked_fill(at::ones({S, S}, q.options().dtype(at::kBool)).triu(1), -INFINITY);
            const Tensor p = at::softmax(score, -1), dp = at::matmul(g, vf.transpose(2, 3).contiguous());
            const Tensor ds = p * (dp - (dp * p).sum(-1, true)) * scale;
            const auto t = q.scalar_type();
            return {at::matmul(ds, kf).to(t), at::matmul(ds.transpose(2, 3).contiguous(), qf).to(t), at::matmul(p.transpose(2, 3).contiguous(), g).to(t), Tensor()};
        }
        const Tensor g = heads_fit(grads[0]) ? grads[0] : dense16(grads[0]);
        Tensor dq = heads_inside(q, B, heads, S, D), dk = heads_inside(q, B, heads, S, D), dv = heads_inside(q, B, heads, S, D), delta = at::empty_like(s[4]);
        const MtsHeads vq = view(q), vk = view(k), vv = view(v), vo = view(s[3]), vg = view(g), vdq = view(dq), vdk = view(dk), vdv = view(dv);
        check(mts_attention_bwd(&vq, &vk, &vv, &vo, &vg, ptr_as<float>(s[4]), B, heads, S, causal, dtype_code(q), &vdq, &vdk, &vdv, ptr_as<float>(delta),
                                stream_of(q)),
              "mts_attention_bwd");
        return {dq, dk, dv, Tensor()};
    }
};

// Rotary encoding and attention of a packed projection [B, S, 3 * heads * 64] as one node: the keys are turned by a launch of their own, the queries
// where the attention reads them, and the gradients are turned back where it writes them, in place in the gradient of the projection.
bool qkv_attention_supported(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t heads) {
    if (!qkv_rope_supported(qkv, cos, sin, heads) || (qkv.scalar_type() != at::kBFloat16 && qkv.scalar_type() != at::kHalf)) return false;
    if (!mts_attention_supported(qkv.size(0), heads, qkv.size(1), qkv.size(2) / (3 * heads)) || !aligned16(cos) || !aligned16(sin)) return false;
    if (at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != qkv.scalar_type()) return false;
    return at::globalContext().userEnabledFlashSDP();
}

struct QkvAttention : torch::autograd::Function<QkvAttention> {
    static MtsHeads view(const Tensor& t) { return {ptr(t), t.stride(0), t.stride(1), t.stride(2)}; }
    // [B, heads, S, D] of queries, keys or values inside a packed projection
    static MtsHeads part(const Tensor& packed, int which, int64_t heads, int64_t D) {
        const int64_t S = packed.size(1), row = packed.size(2);
        return {static_cast<char*>(ptr(packed)) + which * heads * D * packed.element_size(), S * row, D, row};
    }
    static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t heads, bool causal, bool backward) {   // dense16
        const int64_t B = qkv.size(0), S = qkv.size(1), D = qkv.size(2) / (3 * heads);
        Tensor k = heads_inside(qkv, B, heads, S, D), q = backward ? heads_inside(qkv, B, heads, S, D) : Tensor();
        Tensor out = at::empty({B, S, heads * D}, qkv.options()), lse = f32({B * heads * S}, qkv);
        launch_rope({{qkv.view({B, S, 3, heads, D}).select(2, 1).transpose(1, 2), k, TURN}}, cos, sin);
        const MtsHeads vq = part(qkv, 0, heads, D), vk = view(k), vv = part(qkv, 2, heads, D), vo = {ptr(out), S * heads * D, D, heads * D};
        const MtsHeads turned = backward ? view(q) : MtsHeads{};
        check(mts_attention_turned_fwd(&vq, &vk, &vv, ptr(cos), ptr(sin), B, heads, S, causal, dtype_code(qkv), backward ? &turned : nullptr, &vo,
                                       ptr_as<float>(lse), stream_of(qkv)),
              "mts_attention_turned_fwd");
        if (backward) {
            ctx->save_for_backward({qkv, q, k, out, lse, cos, sin});
            ctx->saved_data["heads"] = heads;
            ctx->saved_data["causal"] = causal;
        }
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &qkv = s[0], &q = s[1], &k = s[2], &cos = s[5], &sin = s[6];
        c10::OptionalDeviceGuard guard(qkv.device());
        const int64_t heads = ctx->saved_data["heads"].toInt(), B = qkv.size(0), S = qkv.size(1), D = qkv.size(2) / (3 * heads);
        const bool causal = ctx->saved_data["causal"].toBool();
        if (written_out(grads)) {   // attention in fp32, as its own node has it
            auto head = [&](const Tensor& t) { return t.view({B, S, heads, D}).transpose(1, 2); };
            const variable_list parts = qkv.chunk(3, -1);
            auto turned = [&](const Tensor& t) {
                const variable_list h = t.chunk(2, -1);
                return t * cos + at::cat({-h[1], h[0]}, -1) * sin;
            };
            const double scale = 1.0 / std::sqrt((double)D);
            const Tensor qf = turned(head(parts[0])).to(at::kFloat), kf = turned(head(parts[1])).to(at::kFloat), vf = head(parts[2]).to(at::kFloat);
            const Tensor g = head(grads[0].contiguous()).to(at::kFloat);
            Tensor score = at::matmul(qf, kf.transpose(2, 3).contiguous()) * scale;
            if (causal) score = score.masked_fill(at::ones({S, S}, qkv.options().dtype(at::kBool)).triu(1), -INFINITY);
            const Tensor p = at::softmax(score, -1), dp = at::matmul(g, vf.transpose(2, 3).contiguous());
            const Tensor ds = p * (dp - (dp * p).sum(-1, true)) * scale;
            auto back = [&](const Tensor& t, bool turn) { return (turn ? turned_back(t.to(qkv.scalar_type()), cos, sin) : t.to(qkv.scalar_type())).transpose(1, 2); };
            const Tensor d = at::stack({back(at::matmul(ds, kf), true), back(at::matmul(ds.transpose(2, 3).contiguous(), qf), true),
                                        back(at::matmul(p.transpose(2, 3).contiguous(), g), false)}, 2);
            return {d.reshape(qkv.sizes()), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
        }
        const Tensor g = dense16(grads[0]), d = at::empty_like(qkv);
        Tensor delta = at::empty_like(s[4]);
        const MtsHeads vq = view(q), vk = view(k), vv = part(qkv, 2, heads, D), rows = {ptr(s[3]), S * heads * D, D, heads * D};
        const MtsHeads vg = {ptr(g), rows.batch_stride, rows.head_stride, rows.row_stride};
        const MtsHeads dq = part(d, 0, heads, D), dk = part(d, 1, heads, D), dv = part(d, 2, heads, D);
        check(mts_attention_turned_bwd(&vq, &vk, &vv, &rows, &vg, ptr_as<float>(s[4]), ptr(cos), ptr(sin), B, heads, S, causal, dtype_code(qkv), &dq, &dk, &dv,
                                       ptr_as<float>(delta), stream_of(qkv)),
              "mts_attention_turned_bwd");
        return {d, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

constexpr int64_t kIgnoreIndex = -100;   // torch's default

bool cross_entropy_supported(const Tensor& logits, const Tensor& targets) {
    return all_plain(logits, targets) && on_one_gpu(logits, targets) && logits.dim() == 2 && targets.dim() == 1 &&
           is_activation_type(logits.scalar_type()) && targets.scalar_type() == at::kLong && logits.size(0) == targets.size(0) && logits.size(0) > 0 && logits.size(0) < MTS_MAX_LOSS_ROWS && logits.size(1) > 0 &&
           logits.size(1) < k2GiB;
}

// Whether gradients of what `fn` made go, through views at most, to a projection whose gradients read rows of any pitch (Linear::in_rounds).  With
// `execution`, the backward pass that is under way: and nobody sees them on the way, by a hook, a retained gradient or as a result of autograd.grad.
bool goes_to_rounds(torch::autograd::Node* fn, const std::unordered_map<torch::autograd::Node*, torch::autograd::GraphTask::ExecInfo>* execution) {
    for (int depth = 0; fn && depth < 4; ++depth) {
        if (!fn->pre_hooks().empty() || !fn->tensor_pre_hooks().empty() || !fn->retains_grad_hooks().empty() || !fn->post_hooks().empty()) return false;
        if (execution) {
            const auto found = execution->find(fn);
            if (found != execution->end() && found->second.captures_) return false;
        }
        if (dynamic_cast<torch::autograd::CppNode<Linear>*>(fn)) return true;
        const std::string name = fn->name();
        if ((name != "ViewBackward0" && name != "UnsafeViewBackward0" && name != "ReshapeAliasBackward0") || fn->num_outputs() != 1) return false;
        fn = fn->next_edge(0).function.get();
    }
    return false;
}
// the same of the gradient that the node `self` returns in this backward pass; whoever sees it gets it dense
bool goes_to_rounds_unseen(torch::autograd::Node* self) {
    const auto* execution = torch::autograd::get_current_graph_task_exec_info();
    return self && execution && self->post_hooks().empty() && goes_to_rounds(self->next_edge(0).function.get(), execution);
}

// mean cross-entropy without an fp32 copy of the logits
struct CrossEntropy : torch::autograd::Function<CrossEntropy> {
    // Whether the gradient is formed with the loss, for a caller who says that the loss is the root of its backward pass (its own gradient is
    // then 1; where it is not after all, the backward pass forms it anew): from logits that are in registers anyway.  Rows as the backward
    // pass will return them, so far as that is known; not where saved tensors are to go elsewhere, and this one would stay.
    static bool formed_ahead(const Tensor& logits) {
        const int64_t V = logits.size(1);
        return at::GradMode::is_enabled() && logits.requires_grad() && mts_cross_entropy_both_supported((int)V, dtype_code(logits)) &&
               !at::SavedTensorDefaultHooks::get_hooks() && (V % 8 == 0 || goes_to_rounds(logits.grad_fn().get(), nullptr));
    }
    // dense16, dense
    static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& targets, bool ahead) {
        const int64_t N = logits.size(0), V = logits.size(1);
        // per row: maximum, log of the sum, loss; then 1 / count.  The loss is a tensor of its own, which the caller may change
        // (no view) and which is not kept.
        Tensor rows = f32({3 * N + 1}, logits), loss = f32({}, logits);
        float* row = ptr_as<float>(rows);
        if (ahead) {
            const int64_t pitch = V % 8 ? row_pitch(V) : V;
            Tensor d = at::empty({N, pitch}, logits.options());
            check(mts_cross_entropy_both(ptr(logits), ptr_as<int64_t>(targets), N, V, kIgnoreIndex, dtype_code(logits), row, row + N, row + 2 * N, ptr_as<float>(loss),
                                         row + 3 * N, ptr(d), pitch, stream_of(logits)),
                  "mts_cross_entropy_both");
            ctx->saved_data["ahead"] = d;
        } else {
            check(mts_cross_entropy_fwd(ptr(logits), ptr_as<int64_t>(targets), N, V, kIgnoreIndex, dtype_code(logits), row, row + N, row + 2 * N,
                                        ptr_as<float>(loss), row + 3 * N, stream_of(logits)),
                  "mts_cross_entropy_fwd");
        }
        ctx->save_for_backward({logits, targets, rows});
        return loss;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        c10::OptionalDeviceGuard guard(s[0].device());
        const int64_t N = s[0].size(0), V = s[0].size(1);
        if (written_out(grads)) {
            const Tensor g = grads[0].to(at::kFloat);
            const Tensor t = s[1].unsqueeze(1), hit = at::arange(V, s[1].options()).unsqueeze(0).eq(t);
            const Tensor p = at::softmax(s[0].to(at::kFloat), 1) - hit.to(at::kFloat), none = at::zeros({}, p.options());
            const Tensor ignored = t.eq(kIgnoreIndex), outside = t.lt(0).logical_or(t.ge(V)).logical_and(ignored.logical_not());
            const Tensor scale = g * s[2].select(0, 3 * N) + at::where(outside, at::full({}, NAN, p.options()), none);
            return {at::where(ignored, none, p * scale).to(s[0].scalar_type()), Tensor(), Tensor()};
        }
        const Tensor g = like_f32(grads[0]);
        const float* row = ptr_as<float>(s[2]);
        const bool pitched = V % 8 && s[0].scalar_type() != at::kFloat && goes_to_rounds_unseen(torch::autograd::get_current_node().get());
        const auto ahead = ctx->saved_data.find("ahead");
        if (ahead != ctx->saved_data.end()) {
            const Tensor rows = ahead->second.toTensor();
            ctx->saved_data.erase(ahead);   // whoever gets it may write to it; a second pass forms its own
            if (V % 8 == 0 || pitched) {
                check(mts_cross_entropy_bwd_unless_one(ptr(s[0]), ptr_as<int64_t>(s[1]), N, V, kIgnoreIndex, dtype_code(s[0]), row, row + N, ptr_as<float>(g),
                                                       row + 3 * N, ptr(rows), rows.size(1), stream_of(s[0])),
                      "mts_cross_entropy_bwd_unless_one");
                return {V % 8 ? rows.narrow(1, 0, V) : rows, Tensor(), Tensor()};
            }
        }
        if (pitched) {
            const int64_t pitch = row_pitch(V);
            Tensor rows = at::empty({N, pitch}, s[0].options());
            check(mts_cross_entropy_bwd_pitched(ptr(s[0]), ptr_as<int64_t>(s[1]), N, V, kIgnoreIndex, dtype_code(s[0]), row, row + N, ptr_as<float>(g),
                                                row + 3 * N, ptr(rows), pitch, stream_of(s[0])),
                  "mts_cross_entropy_bwd_pitched");
            return {rows.narrow(1, 0, V), Tensor(), Tensor()};
        }
        Tensor d = at::empty_like(s[0]);
        check(mts_cross_entropy_bwd(ptr(s[0]), ptr_as<int64_t>(s[1]), N, V, kIgnoreIndex, dtype_code(s[0]), row, row + N, ptr_as<float>(g),
                                    row + 3 * N, ptr(d), stream_of(s[0])),
              "mts_cross_entropy_bwd");
        return {d, Tensor(), Tensor()};
    }
};

// ---- numbers of a model's layers -----------------------------------------------------------------------------------------------

typedef std::vector<std::vector<Tensor>> Groups;   // tensors of one quantity, one a layer

// `differentiable` groups come first; the others carry no gradient
bool layer_means_supported(const Groups& groups, int64_t differentiable) {
    if (groups.empty() || groups.size() > MTS_MEAN_GROUPS || groups[0].empty() || !nobody_dispatches() || at::impl::torch_function_mode_enabled()) return false;
    size_t tensors = 0;
    const at::Device device = groups[0][0].device();
    for (size_t g = 0; g < groups.size(); ++g) {
        if (groups[g].empty()) return false;
        const Tensor& first = groups[g][0];
        const bool tracked = (int64_t)g < differentiable;
        if (tracked ? first.dim() != 0 : first.dim() > 1) return false;
        if (first.numel() < 1 || !(first.scalar_type() == at::kFloat || (first.scalar_type() == at::kLong && first.dim() == 0 && !tracked))) return false;
        for (const Tensor& t : groups[g])
            if (!is_plain(t) || !t.is_cuda() || t.device() != device || t.scalar_type() != first.scalar_type() || t.sizes() != first.sizes() || !t.is_contiguous() ||
                (!tracked && t.requires_grad()))
                return false;
        tensors += groups[g].size();
    }
    return tensors <= MTS_MEAN_TENSORS;
}

void scalar_sums(std::initializer_list<Tensor> in, const float (&weight)[4][4], const int (&terms)[4], const float (&divisor)[4],
                 std::initializer_list<Tensor> out) {
    const float* sources[4] = {};
    float* results[4] = {};
    int inputs = 0, outputs = 0;
    for (const Tensor& t : in) sources[inputs++] = ptr_as<float>(t);
    for (const Tensor& t : out) results[outputs++] = ptr_as<float>(t);
    check(mts_scalar_sums(sources, inputs, &weight[0][0], terms, divisor, results, outputs, stream_of(*out.begin())), "mts_scalar_sums");
}

// The mean of every group, fp32.  `tracked`: the tensors of the differentiable groups, for autograd.
struct LayerMeans : torch::autograd::Function<LayerMeans> {
    static variable_list means(const Groups& groups, int64_t differentiable) {
        const void* src[MTS_MEAN_TENSORS];
        int first[MTS_MEAN_GROUPS + 1] = {}, n[MTS_MEAN_GROUPS], whole[MTS_MEAN_GROUPS];
        float* out[MTS_MEAN_GROUPS];
        int64_t total = 0;
        for (size_t g = differentiable; g < groups.size(); ++g) total += groups[g][0].numel();
        const Tensor& like = groups[0][0];
        const Tensor records = f32({std::max<int64_t>(total, 1)}, like);
        variable_list result;
        int64_t at_element = 0;
        for (size_t g = 0; g < groups.size(); ++g) {
            const Tensor& t = groups[g][0];
            if ((int64_t)g < differentiable) result.push_back(f32({}, like));
            else {
                result.push_back(part_of(records, at_element * 4, t.sizes(), at::kFloat));
                at_element += t.numel();
            }
            first[g + 1] = first[g] + (int)groups[g].size(), n[g] = (int)t.numel(), whole[g] = t.scalar_type() == at::kLong, out[g] = ptr_as<float>(result.back());
            for (size_t l = 0; l < groups[g].size(); ++l) src[first[g] + l] = ptr(groups[g][l]);
        }
        check(mts_layer_means(src, first, n, whole, (int)groups.size(), out, stream_of(like)), "mts_layer_means");
        return result;
    }
    static variable_list forward(AutogradContext* ctx, at::TensorList tracked, const Groups& groups, int64_t differentiable) {
        variable_list result = means(groups, differentiable);
        std::vector<int64_t> counts;
        for (int64_t g = 0; g < differentiable; ++g) counts.push_back((int64_t)groups[g].size());
        ctx->saved_data["counts"] = counts;
        ctx->mark_non_differentiable(variable_list(result.begin() + differentiable, result.end()));
        ctx->set_materialize_grads(false);
        return result;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto counts = ctx->saved_data["counts"].toIntVector();
        const bool stock = written_out(grads);
        variable_list result;
        Tensor share[2];
        if (!stock && counts.size() == 2 && grads[0].defined() && grads[1].defined()) {
            c10::OptionalDeviceGuard guard(grads[0].device());
            for (Tensor& t : share) t = f32({}, grads[0]);
            const Tensor a = grads[0].to(at::kFloat), b = grads[1].to(at::kFloat);
            scalar_sums({a, b}, {{1.f, 0.f}, {0.f, 1.f}}, {1, 2}, {(float)counts[0], (float)counts[1]}, {share[0], share[1]});
        }
        for (size_t g = 0; g < counts.size(); ++g) {
            const Tensor one = !grads[g].defined() ? Tensor() : g < 2 && share[g].defined() ? share[g] : grads[g] / (double)counts[g];
            result.insert(result.end(), (size_t)counts[g], one);
        }
        result.resize(result.size() + 2);
        return result;
    }
};

bool total_loss_supported(const Tensor& loss, const Tensor& aux, const Tensor& z) {
    auto number = [](const Tensor& t) { return t.dim() == 0 && t.scalar_type() == at::kFloat; };
    return all_plain(loss, aux, z) && on_one_gpu(loss, aux, z) && number(loss) && number(aux) && number(z);
}

// loss + a * aux + b * z; and without a gradient a * aux, b * z and the sum of the two
struct TotalLoss : torch::autograd::Function<TotalLoss> {
    static variable_list forward(AutogradContext* ctx, const Tensor& loss, const Tensor& aux, const Tensor& z, double a, double b) {
        Tensor total = f32({}, loss), parts = f32({3}, loss);
        auto part = [&](int i) { return part_of(parts, i * 4, {}, at::kFloat); };
        const variable_list out{total, part(0), part(1), part(2)};
        const float fa = (float)a, fb = (float)b;
        scalar_sums({loss, aux, z}, {{1.f, fa, fb}, {0.f, fa, 0.f}, {0.f, 0.f, fb}, {0.f, fa, fb}}, {7, 2, 4, 6}, {1.f, 1.f, 1.f, 1.f}, {out[0], out[1], out[2], out[3]});
        ctx->saved_data["a"] = a;
        ctx->saved_data["b"] = b;
        ctx->mark_non_differentiable({out[1], out[2], out[3]});
        ctx->set_materialize_grads(false);
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const Tensor& g = grads[0];
        const double a = ctx->saved_data["a"].toDouble(), b = ctx->saved_data["b"].toDouble();
        if (!g.defined()) return variable_list(5);
        if (written_out(grads) || g.scalar_type() != at::kFloat) return {g, g * a, g * b, Tensor(), Tensor()};
        c10::OptionalDeviceGuard guard(g.device());
        Tensor d_aux = f32({}, g), d_z = f32({}, g);
        scalar_sums({g}, {{(float)a}, {(float)b}}, {1, 1}, {1.f, 1.f}, {d_aux, d_z});
        return {g, d_aux, d_z, Tensor(), Tensor()};
    }
};

// ---- optimizer update ------------------------------------------------------------------------------------------------------------

// Whether one update may be taken by the kernels: fp32 parameters, dense gradients and moments on one GPU, a step count on it for each.
bool adamw_supported(const std::vector<Tensor>& params, const std::vector<Tensor>& exp_avgs, const std::vector<Tensor>& exp_avg_sqs,
                     const std::vector<Tensor>& steps) {
    if (params.empty() || exp_avgs.size() != params.size() || exp_avg_sqs.size() != params.size() || steps.size() != params.size() ||
        params.size() >= (1u << 20) || !nobody_dispatches())
        return false;
    auto fits = [&](const Tensor& t, const Tensor& p) {
        return t.defined() && is_plain(t) && t.layout() == at::kStrided && t.scalar_type() == at::kFloat && t.device() == params[0].device() &&
               t.is_contiguous() && t.sizes() == p.sizes();
    };
    for (size_t i = 0; i < params.size(); ++i) {
        const Tensor &p = params[i], &step = steps[i];
        if (!p.is_cuda() || !fits(p, p) || !fits(p.grad(), p) || !fits(exp_avgs[i], p) || !fits(exp_avg_sqs[i], p) || p.numel() >= (1LL << 30)) return false;
        if (!is_plain(step) || step.layout() != at::kStrided || step.device() != p.device() || step.scalar_type() != at::kFloat || step.numel() != 1) return false;
    }
    return true;
}

// norm of the gradients, clipping coefficient, and whether norm or loss are not finite; max_norm < 0: the gradients stay out of it
Tensor grad_norm(const std::vector<Tensor>& params, double max_norm, const Tensor& loss) {
    std::vector<MtsGradSpan> spans;
    if (max_norm >= 0)
        for (const Tensor& p : params) spans.push_back({ptr_as<float>(p.grad()), p.numel()});
    Tensor result = f32({3}, params[0]);
    const int64_t ws_bytes = mts_grad_norm_workspace_bytes(spans.data(), (int)spans.size());
    Tensor ws = bytes(ws_bytes, params[0]);
    check(mts_grad_norm(spans.data(), (int)spans.size(), (float)max_norm, ptr_as<float>(loss), ptr_as<float>(result), ptr(ws), ws.numel(), stream_of(params[0])),
          "mts_grad_norm");
    return result;
}

// groups: of each tensor; settings: lr, beta1, beta2, eps and weight decay of each group; scale: what grad_norm returned, clipped: from the gradients
void adamw(const std::vector<Tensor>& params, const std::vector<Tensor>& exp_avgs, const std::vector<Tensor>& exp_avg_sqs, const std::vector<Tensor>& steps,
           const std::vector<int64_t>& groups, const std::vector<std::array<double, 5>>& settings, const Tensor& scale, bool clipped, bool skip_if_not_finite) {
    std::vector<MtsAdamTensor> tensors;
    std::vector<Tensor> held;   // gradients that somebody else holds: left clipped, and marked as written, as stock clipping leaves them
    for (size_t i = 0; i < params.size(); ++i) {
        const Tensor& g = params[i].grad();
        const bool keep = clipped && (g.use_count() > 1 || g.storage().use_count() > 1);
        tensors.push_back({ptr_as<float>(params[i]), ptr_as<float>(g), ptr_as<float>(exp_avgs[i]), ptr_as<float>(exp_avg_sqs[i]), ptr_as<float>(steps[i]),
                           params[i].numel(), (int)groups[i], keep});
        if (keep) held.push_back(g);
    }
    std::vector<MtsAdamGroup> of;
    for (const auto& s : settings) of.push_back({s[0], s[1], s[2], s[3], s[4]});
    Tensor ws = bytes(mts_adamw_workspace_bytes((int)tensors.size()), params[0]);
    const float* result = ptr_as<float>(scale);
    check(mts_adamw(tensors.data(), (int)tensors.size(), of.data(), (int)of.size(), result + 1, skip_if_not_finite ? result + 2 : nullptr, ptr(ws), ws.numel(),
                    stream_of(params[0])),
          "mts_adamw");
    // The stock fused operator marks neither parameters nor state as written: graphs that have saved one go on.
    for (const Tensor& g : held)
        if (!g.is_inference()) g.unsafeGetTensorImpl()->bump_version();
}

}  // namespace

PYBIND11_MODULE(_host, m) {
    namespace py = pybind11;
    m.def("set_joint_workspace", [](py::object f) { joint_workspace_of = new py::object(std::move(f)); });
    m.def("fused_moe_violation", &fused_moe_violation);
    m.def("layer_violation", &layer_violation);
    m.def("needs_padding", &needs_padding);
    m.def("router_logits_supported", &router_logits_supported);
    m.def("route", [](const Tensor& index, int64_t E) {
        const Routing r = route(index.contiguous(), E);
        return std::make_tuple(r.expert_start, r.x_gather, r.s_scatter, r.s_reverse);
    });
    m.def("fused_moe", [](const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& index, const Tensor& weights, int64_t switches, int64_t limit) {
        c10::OptionalDeviceGuard guard(x.device());
        return FusedMoE::apply(x, w1, w2, index, weights, switches | no_backward(x, w1, w2, weights), limit);
    });
    m.def("moe_layer", [](const Tensor& x, const Tensor& w_r, const Tensor& w1, const Tensor& w2, int64_t top_k, bool normalize, int64_t capacity, int64_t switches,
                          int64_t limit) {
        c10::OptionalDeviceGuard guard(x.device());
        const int64_t without = no_backward(x, w_r, w1, w2);
        if (without && all_plain(x, w_r, w1, w2)) {   // no node
            const LayerForward f = layer_forward(x, w_r, w1, w2, top_k, normalize, capacity, {switches | without, limit});
            return std::make_tuple(f.out, f.load_balance, f.z_loss, f.prob_mean, f.entropy, f.counts, f.load_stats, f.indices, f.weights);
        }
        const variable_list v = MoELayer::apply(x, w_r, w1, w2, top_k, normalize, capacity, switches | without, limit);
        return std::make_tuple(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8]);
    });
    m.def("router_postprocess", [](const Tensor& logits, int64_t top_k, bool normalize, int64_t act_dtype) {
        c10::OptionalDeviceGuard guard(logits.device());
        return RouterPostprocess::apply(logits, top_k, normalize, act_dtype);
    });
    m.def("router_logits", [](const Tensor& x, const Tensor& w) {
        c10::OptionalDeviceGuard guard(x.device());
        return RouterLogits::apply(dense_router_operand(x, w.size(0)), dense_router_operand(w, w.size(0)));
    });
    m.def("rmsnorm_supported", &rmsnorm_supported);
    m.def("rmsnorm", [](const Tensor& x, const Tensor& w, double eps) {
        c10::OptionalDeviceGuard guard(x.device());
        return RMSNorm::apply(dense16(x), MaybeTensor(), dense16(w), eps)[0];
    });
    m.def("add_rmsnorm", [](const Tensor& x, const Tensor& residual, const Tensor& w, double eps) {
        c10::OptionalDeviceGuard guard(x.device());
        const variable_list v = RMSNorm::apply(dense16(x), MaybeTensor(dense16(residual)), dense16(w), eps);
        return std::make_tuple(v[0], v[1]);
    });
    m.def("rope_supported", &rope_supported);
    m.def("rope", [](const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin) {
        c10::OptionalDeviceGuard guard(q.device());
        const variable_list v = Rope::apply(q, k, cos, sin);
        return std::make_tuple(v[0], v[1]);
    });
    m.def("qkv_rope_supported", &qkv_rope_supported);
    m.def("qkv_rope", [](const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t heads) {
        c10::OptionalDeviceGuard guard(qkv.device());
        const variable_list v = QkvRope::apply(qkv, cos, sin, heads);
        return std::make_tuple(v[0], v[1], v[2]);
    });
    m.def("linear_supported", &linear_supported);
    m.def("linear_rows_fit", &rows_fit);
    m.def("linear", [](const Tensor& x, const Tensor& w) {
        c10::OptionalDeviceGuard guard(x.device());
        return Linear::apply(x, w);
    });
    m.def("linear_alone_supported", &linear_alone_supported);
    m.def("linear_alone", [](const Tensor& x, const Tensor& w) {
        c10::OptionalDeviceGuard guard(x.device());
        return linear_alone(x, w);
    });
    m.def("embedding_supported", &embedding_supported);
    m.def("embedding", [](const Tensor& ids, const Tensor& w, at::ScalarType type) {
        c10::OptionalDeviceGuard guard(w.device());
        return Embedding::apply(ids, w, type);
    });
    m.def("attention_supported", &attention_supported);
    m.def("attention", [](const Tensor& q, const Tensor& k, const Tensor& v, bool causal) {
        c10::OptionalDeviceGuard guard(q.device());
        return Attention::apply(q, k, v, causal);
    });
    m.def("qkv_attention_supported", &qkv_attention_supported);
    m.def("qkv_attention", [](const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t heads, bool causal) {
        c10::OptionalDeviceGuard guard(qkv.device());
        return QkvAttention::apply(dense16(qkv), cos, sin, heads, causal, at::GradMode::is_enabled() && qkv.requires_grad());
    });
    m.def("layer_means_supported", &layer_means_supported);
    m.def("layer_means", [](const Groups& groups, int64_t differentiable) {
        c10::OptionalDeviceGuard guard(groups.at(0).at(0).device());
        variable_list tracked;
        bool wanted = false;
        for (int64_t g = 0; g < differentiable; ++g)
            for (const Tensor& t : groups.at(g)) {
                tracked.push_back(t);
                wanted |= t.requires_grad();
            }
        if (!wanted || !at::GradMode::is_enabled()) return LayerMeans::means(groups, differentiable);
        return LayerMeans::apply(at::TensorList(tracked), groups, differentiable);
    });
    m.def("total_loss_supported", &total_loss_supported);
    m.def("total_loss", [](const Tensor& loss, const Tensor& aux, const Tensor& z, double a, double b) {
        c10::OptionalDeviceGuard guard(loss.device());
        const variable_list v = TotalLoss::apply(loss, aux, z, a, b);
        return std::make_tuple(v[0], v[1], v[2], v[3]);
    });
    m.attr("ADAM_GROUPS") = MTS_ADAM_GROUPS;
    // not by way of Python's `grad`, whose object counts as a holder of the gradient from then on
    m.def("gradients_defined", [](const std::vector<Tensor>& params) {
        std::vector<bool> defined;
        for (const Tensor& p : params) defined.push_back(p.grad().defined());
        return defined;
    });
    m.def("drop_gradients", [](const std::vector<Tensor>& params) {
        for (const Tensor& p : params) p.mutable_grad().reset();
    });
    m.def("adamw_supported", &adamw_supported);
    m.def("grad_norm", [](const std::vector<Tensor>& params, double max_norm, const Tensor& loss) {
        c10::OptionalDeviceGuard guard(params.at(0).device());
        return grad_norm(params, max_norm, loss);
    });
    m.def("adamw", [](const std::vector<Tensor>& params, const std::vector<Tensor>& exp_avgs, const std::vector<Tensor>& exp_avg_sqs,
                      const std::vector<Tensor>& steps, const std::vector<int64_t>& groups, const std::vector<std::array<double, 5>>& settings, const Tensor& scale,
                      bool clipped, bool skip_if_not_finite) {
        c10::OptionalDeviceGuard guard(params.at(0).device());
        adamw(params, exp_avgs, exp_avg_sqs, steps, groups, settings, scale, clipped, skip_if_not_finite);
    });
    m.def("cross_entropy_supported", &cross_entropy_supported);
    m.def("cross_entropy", [](const Tensor& logits, const Tensor& targets, bool is_root) {
        c10::OptionalDeviceGuard guard(logits.device());
        const Tensor dense = dense16(logits);
        return CrossEntropy::apply(dense, targets.contiguous(), is_root && CrossEntropy::formed_ahead(dense));
    });
}
