// Host path of the ops: argument checks, output / workspace allocation, kernel launches through the
// C ABI and the autograd nodes, as a CPython extension module (slapo_amd/_host.so).
//
// Why native: a training step calls these ops hundreds of times and most calls are shorter than the
// host work around them.  With torch.autograd.Function and ctypes a forward + backward pair cost
// 100-175 us of Python on the launching and the engine thread whatever the kernels took (fp16
// 1537 x 768 bias + dropout + residual + LayerNorm: 175-187 us per pair against 22 us of kernels).
// The nodes here derive from torch::autograd::Node directly: the backward runs on the engine's
// thread without the interpreter lock, and a call allocates its outputs and nothing else.
//
// Nothing in this file computes: every number comes from a kernel behind include/slapo_amd.h.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <ATen/core/Generator.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

#include "../../include/slapo_amd.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---- errors -------------------------------------------------------------------------------------

// A negative status of the C ABI becomes the exception that slapo_amd._lib.check raises.
void check(int status, const char* what) {
    if (status == SLAPO_OK) return;
    const std::string text = std::string(what) + " failed: " + slapo_amd_status_string(status) +
                             " (status " + std::to_string(status) + ")";
    if (status >= SLAPO_ERR_ARG) TORCH_CHECK_VALUE(false, text);
    pybind11::gil_scoped_acquire gil;
    PyObject* mod = PyImport_ImportModule("slapo_amd._lib");
    PyObject* cls = mod ? PyObject_GetAttrString(mod, "SlapoAmdError") : nullptr;
    if (cls) PyErr_SetString(cls, text.c_str());
    Py_XDECREF(cls);
    Py_XDECREF(mod);
    python_error err;
    err.persist();
    throw std::move(err);
}

void require_device(std::initializer_list<const Tensor*> tensors) {
    for (const Tensor* t : tensors)
        if (t->defined() && !t->is_cuda())
            TORCH_CHECK(false,
                        "slapo_amd kernels run on a gfx950 device only; got a tensor on '",
                        t->device().str(),
                        "'.  There is no CPU implementation in this package.");
}

// Tangents of forward-mode differentiation would be dropped without a word: refuse them, as
// torch.autograd.Function does for a function without `jvp`.
void refuse_tangents(std::initializer_list<const Tensor*> tensors) {
    for (const Tensor* t : tensors)
        if (t->defined() && t->_fw_grad(0).defined())
            TORCH_CHECK(false, "slapo_amd ops do not implement forward-mode differentiation");
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return SLAPO_F32;
        case at::kHalf: return SLAPO_F16;
        case at::kBFloat16: return SLAPO_BF16;
        default:
            TORCH_CHECK_VALUE(false, "unsupported dtype ", t,
                              "; expected float32, float16 or bfloat16");
    }
}

// ---- small helpers ------------------------------------------------------------------------------

void* stream_of(const Tensor& t) {
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}
bool capturing() {
    return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

const void* cptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* mptr(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0; }

// An uninitialised contiguous tensor on the current device, straight from torch's caching allocator:
// at::empty takes twice as long (1.7 us) to get there, and a training step makes hundreds.
Tensor fresh(at::IntArrayRef sizes, at::ScalarType dtype) {
    static c10::Allocator* const allocator = at::detail::getCUDAHooks().getCUDADeviceAllocator();
    return at::detail::empty_generic(sizes, allocator, c10::DispatchKeySet(c10::DispatchKey::CUDA),
                                     dtype, std::nullopt);
}
Tensor fresh_like(const Tensor& t) { return fresh(t.sizes(), t.scalar_type()); }
Tensor floats(int64_t n) { return fresh({n > 0 ? n : 1}, at::kFloat); }

Tensor cast(const Tensor& t, at::ScalarType dt) {
    return !t.defined() || t.scalar_type() == dt ? t : t.to(dt);
}
// contiguous and of dtype `dt`
Tensor dense(const Tensor& t, at::ScalarType dt) {
    return t.defined() ? cast(t.contiguous(), dt) : t;
}

// What saved-tensor hooks hand back has the values of what was saved; the kernels need it dense too.
Tensor unpack_dense(const SavedVariable& s, std::shared_ptr<Node> owner = nullptr) {
    const Tensor t = s.unpack(std::move(owner));
    return t.defined() ? t.contiguous() : t;
}
SavedVariable keep(const Tensor& t, bool is_output = false) {
    return t.defined() ? SavedVariable(t, is_output) : SavedVariable();
}

// Dropout of one call: probability, the (seed, offset) pair drawn for it -- by value, or in the
// device memory of `state` while a graph is being captured -- and the launch plan.
struct Dropout {
    double p = 0.0;
    uint64_t seed = 0, offset = 0;
    Tensor state;
    slapo_dropout_plan plan = {};

    const slapo_dropout_plan* plan_ptr() const { return p > 0.0 ? &plan : nullptr; }
    void set_plan(int64_t numel, int elem_bytes, const at::Device& dev) {
        if (!(p > 0.0)) return;
        check(slapo_amd_dropout_plan(numel, elem_bytes, 256, dev.index(), &plan),
              "slapo_amd_dropout_plan");
        if (state.defined()) {
            TORCH_CHECK_VALUE(
                state.is_cuda() && state.numel() == 2 && state.is_contiguous() &&
                    (state.scalar_type() == at::kLong || state.scalar_type() == at::kUInt64),
                "rng_state must be a contiguous device tensor of two 64-bit integers");
            plan.rng_state = state.const_data_ptr();
        }
    }
};

template <typename T, typename... Inputs>
std::shared_ptr<T> make_node(bool wanted, const Inputs&... inputs) {
    if (!wanted) return nullptr;
    std::shared_ptr<T> node(new T(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(inputs...));
    return node;
}

// ---- attention ----------------------------------------------------------------------------------

// wanted: batch, heads, seqlen_q, seqlen_k
void check_mask(const Tensor& mask, const std::array<int64_t, 4>& wanted) {
    if (!mask.defined()) return;
    TORCH_CHECK_VALUE(mask.dim() == 4, "attention_mask must be 4-D ([B,1,1,Sk] or [B,H,Sq,Sk])");
    for (int i = 0; i < 4; ++i)
        TORCH_CHECK(mask.size(i) == wanted[i] || mask.size(i) == 1, "attention_mask of shape ",
                    mask.sizes(), " does not broadcast to ", at::IntArrayRef(wanted));
}

struct AttnProblem {
    slapo_attn_params prm = {};
    Tensor bias;  // of type bias_type, addressed with prm.bias_strides (0 on broadcast dims)
    int bias_type = SLAPO_F32;
    // The fp32 mask that `bias` was prepared from: what the backward keeps and prepares again, as
    // the calls that share a mask would otherwise hold an fp32 copy of it each (fp16 B21 S1512 H11
    // D72, four layers: 1004 -> 207 MB, forward + backward 1.12 -> 1.21 ms).  Other types need an
    // fp32 copy per call anyway.
    Tensor prepared_from;
    Dropout drop;
    at::ScalarType dtype = at::kFloat;

    int64_t b() const { return prm.batch; }
    int64_t h() const { return prm.heads; }
    int64_t sq() const { return prm.seqlen_q; }
    int64_t sk() const { return prm.seqlen_k; }
    int64_t d() const { return prm.head_dim; }
    bool empty() const { return b() * h() * sq() * d() == 0; }

    void describe(at::ScalarType type, int64_t b, int64_t sq, int64_t sk, int64_t h, int64_t d,
                  bool causal, int64_t window, std::optional<double> scale) {
        dtype = type;
        prm.dtype = dtype_code(dtype);
        prm.batch = (int32_t)b, prm.heads = (int32_t)h, prm.head_dim = (int32_t)d;
        prm.seqlen_q = (int32_t)sq, prm.seqlen_k = (int32_t)sk;
        prm.causal = causal ? 1 : 0;
        prm.window = (int32_t)window;
        prm.scale = (float)(scale ? *scale : 1.0 / std::sqrt((double)d));
    }
    // The strides of a mask that is read as it is, 0 on broadcast dims.  Also of the one that the
    // backward gets back: saved-tensor hooks keep its values, not its layout.
    void address_bias() {
        const int64_t wanted[4] = {b(), h(), sq(), sk()};
        for (int i = 0; i < 4; ++i)
            prm.bias_strides[i] = bias.size(i) == 1 && wanted[i] != 1 ? 0 : bias.stride(i);
    }
    // Additive mask, broadcast dims with stride 0.  The fp32 kernels read any layout and type.  The
    // 16-bit ones read one value per key, in the mask's own type at inference (no backward to follow,
    // no dropout); a
    // mask with values per query is prepared for them -- a pass over it that replaces the
    // conversion to fp32 -- unless it is fp32 already and every (batch, head) has values of its
    // own: then it is read once per direction, in place.
    void set_bias(const Tensor& mask, bool infer) {
        if (!mask.defined()) return;
        check_mask(mask, {b(), h(), sq(), sk()});
        const at::ScalarType mt = mask.scalar_type();
        const bool known = mt == at::kFloat || mt == at::kHalf || mt == at::kBFloat16;
        const bool per_key = mask.size(2) == 1;
        bias = known && (infer || !per_key || dtype == at::kFloat) ? mask : cast(mask, at::kFloat);
        bias_type = dtype_code(bias.scalar_type());
        // (the 16-bit kernels address a row of 16-bit values with 32-bit offsets)
        if (bias_type != SLAPO_F32 && per_key && dtype != at::kFloat && bias.size(3) > 1 &&
            bias.stride(3) * sk() >= int64_t(1) << 30)
            bias = bias.contiguous();
        address_bias();
        if (dtype == at::kFloat || per_key || empty() || sk() == 0) return;
        const int64_t mb = prm.bias_strides[0] ? b() : 1, mh = prm.bias_strides[1] ? h() : 1;
        const int64_t bytes =
            (int64_t)slapo_amd_attn_prepared_bias_bytes(mb, mh, sq(), sk());
        if (bytes == 0 || (bias_type == SLAPO_F32 && mb * mh == b() * h())) {
            bias = cast(bias, at::kFloat);
            address_bias();
            bias_type = SLAPO_F32;
            return;
        }
        const Tensor rows = fresh({bytes / 4}, at::kFloat);
        check(slapo_amd_attn_prepare_bias(cptr(bias), bias_type, prm.bias_strides, mb, mh, sq(),
                                          sk(), static_cast<float*>(mptr(rows)), stream_of(bias)),
              "slapo_amd_attn_prepare_bias");
        if (mask.scalar_type() == at::kFloat) prepared_from = mask;
        bias = rows;
        bias_type = SLAPO_BIAS_PREPARED;
        const int64_t pitch = (sk() + 63) / 64 * 64, plane = (sq() + 63) / 64 * 64 * pitch;
        prm.bias_strides[0] = mb > 1 ? mh * plane : 0;
        prm.bias_strides[1] = mh > 1 ? plane : 0;
        prm.bias_strides[2] = pitch;
        prm.bias_strides[3] = 1;
    }
    // Draws, once the geometry is known: F.dropout leaves the generator alone for an empty tensor.
    void set_dropout(Dropout&& in, const at::Device& dev) {
        drop = std::move(in);
        const int64_t scores = b() * h() * sq() * sk();
        if (scores == 0) drop.p = 0.0;
        drop.set_plan(scores, 4, dev);
        prm.p_drop = (float)drop.p;
        prm.seed = drop.seed;
        prm.offset = drop.offset;
        if (drop.p > 0.0) prm.plan = drop.plan;
    }
};

void check_operands(const Tensor& q, const Tensor& k, const Tensor& v) {
    TORCH_CHECK_VALUE(q.dim() == 4 && k.dim() == 4 && v.dim() == 4,
                      "q, k, v must be [batch, seqlen, heads, head_dim]");
    TORCH_CHECK_VALUE(k.sizes() == v.sizes() && q.size(0) == k.size(0) && q.size(2) == k.size(2) &&
                          q.size(3) == k.size(3),
                      "inconsistent q/k/v shapes ", q.sizes(), " ", k.sizes(), " ", v.sizes());
    TORCH_CHECK_VALUE(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(),
                      "q, k, v must share a dtype");
    require_device({&q, &k, &v});
}

void check_packed(const Tensor& qkv, int64_t head_dim) {
    TORCH_CHECK_VALUE(qkv.dim() == 3 && head_dim > 0 && qkv.size(2) % (3 * head_dim) == 0,
                      "qkv must be [batch, seqlen, heads * 3 * head_dim]");
}

// A mask receives no gradient: what is saved of it must not hold on to how it was computed.
Tensor detached(const Tensor& t) { return t.defined() && t.requires_grad() ? t.detach() : t; }

struct AttnResult {
    Tensor out, lse, keep_mask;
};

// The three operands of a call: tensors of their own, or views of one packed [B, S, H, 3 D] tensor.
struct Operands {
    Tensor t[3];
    const void* ptr[3] = {nullptr, nullptr, nullptr};
    bool packed = false;

    void take(AttnProblem& a, const Tensor& q, const Tensor& k, const Tensor& v) {
        const Tensor* in[3] = {&q, &k, &v};
        int64_t* strides[3] = {a.prm.q_strides, a.prm.k_strides, a.prm.v_strides};
        for (int i = 0; i < 3; ++i) {
            t[i] = usable(*in[i]);
            ptr[i] = cptr(t[i]);
            for (int j = 0; j < 3; ++j) strides[i][j] = t[i].stride(j);
        }
    }
    void take_packed(AttnProblem& a, const Tensor& qkv) {
        packed = true;
        t[0] = qkv.contiguous();
        if (!aligned(t[0])) t[0] = t[0].clone();
        packed_views(a, cptr(t[0]), ptr, a.prm.q_strides, a.prm.k_strides, a.prm.v_strides);
    }
    // q, k, v (or their gradients) inside a dense packed buffer
    template <typename P>
    static void packed_views(const AttnProblem& a, P* base, P* (&at)[3], int64_t* qs, int64_t* ks,
                             int64_t* vs) {
        const int64_t esz = a.prm.dtype == SLAPO_F32 ? 4 : 2, row = 3 * a.h() * a.d();
        const int64_t st[3] = {a.sq() * row, row, 3 * a.d()};
        for (int64_t* s : {qs, ks, vs}) std::memcpy(s, st, sizeof st);
        typedef std::conditional_t<std::is_const<P>::value, const char, char> byte;
        for (int i = 0; i < 3; ++i)
            at[i] = base ? reinterpret_cast<byte*>(base) + i * a.d() * esz : nullptr;
    }

 private:
    // Strided [B, S, H, D] views are read as they are while their rows stay 16-byte aligned.
    static Tensor usable(const Tensor& in) {
        const auto st = in.strides();
        bool ok = in.size(3) <= 1 || st[3] == 1;
        if (ok) {
            const int64_t esz = in.element_size();
            ok = aligned(in) && st[0] * esz % 16 == 0 && st[1] * esz % 16 == 0 &&
                 st[2] * esz % 16 == 0;
        }
        return ok ? in : in.contiguous();
    }
};

AttnResult launch_attn_fwd(AttnProblem& a, const Operands& x, at::IntArrayRef out_sizes,
                           bool save_mask, int64_t save_mask_max) {
    AttnResult r;
    slapo_attn_params& prm = a.prm;
    r.out = fresh(out_sizes, a.dtype);
    r.lse = fresh({a.b(), a.h(), a.sq()}, at::kFloat);
    prm.o_strides[0] = a.sq() * a.h() * a.d();
    prm.o_strides[1] = a.h() * a.d();
    prm.o_strides[2] = a.d();
    if (a.empty()) return r;
    if (save_mask) {
        const int64_t bytes = (int64_t)slapo_amd_attn_keep_mask_bytes(&prm);
        if (bytes > 0 && bytes <= save_mask_max) {
            r.keep_mask = fresh({bytes / 4}, at::kInt);
            prm.keep_mask = r.keep_mask.mutable_data_ptr();
        }
    }
    const size_t ws_bytes =
        slapo_amd_attn_fwd_workspace_bytes_for(&prm, a.bias.defined() ? a.bias_type : SLAPO_BIAS_NONE);
    const Tensor ws = ws_bytes ? floats((int64_t)(ws_bytes / 4)) : Tensor();
    check(slapo_amd_attn_fwd_ex(&prm, x.ptr[0], x.ptr[1], x.ptr[2], cptr(a.bias), a.bias_type,
                                mptr(r.out), static_cast<float*>(mptr(r.lse)), mptr(ws), ws_bytes,
                                stream_of(r.out)),
          "slapo_amd_attn_fwd_ex");
    return r;
}

// dst, ds: where dq / dk / dv go and their three outer strides.
void launch_attn_bwd(AttnProblem& a, const Operands& x, const Tensor& out, const Tensor& lse,
                     const Tensor& keep_mask, const Tensor& grad, void* const (&dst)[3],
                     const int64_t (&ds)[3][3]) {
    Tensor dout = cast(grad, a.dtype).contiguous();
    if (!aligned(dout)) dout = dout.clone();
    a.prm.keep_mask = mptr(keep_mask);
    const size_t ws_bytes = slapo_amd_attn_bwd_ex_workspace_bytes_for(
        &a.prm, a.bias.defined() ? a.bias_type : SLAPO_BIAS_NONE);
    const Tensor ws = floats((int64_t)(ws_bytes / 4));
    check(slapo_amd_attn_bwd_ex(&a.prm, x.ptr[0], x.ptr[1], x.ptr[2], cptr(a.bias), a.bias_type,
                                cptr(out), cptr(dout), static_cast<const float*>(cptr(lse)),
                                dst[0], dst[1], dst[2], ds[0], ds[1], ds[2], mptr(ws), ws_bytes,
                                stream_of(out)),
          "slapo_amd_attn_bwd_ex");
}

// Forward saves q, k, v (or the packed tensor), bias, out, lse, the (seed, offset) pair and, with
// dropout, the keep bits; the backward recomputes the probabilities from lse and reads (or
// regenerates) the dropout mask -- it never draws.  The gradient of a packed tensor is written in
// place as three strided views: no concatenation afterwards.
struct AttnBackward : Node {
    AttnProblem a;
    SavedVariable x[3], bias, out, lse, keep_mask, state;
    bool packed = false, prepare = false;  // prepare: `bias` is the mask itself

    std::string name() const override { return "HipAttentionBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* s : {&x[0], &x[1], &x[2], &bias, &out, &lse, &keep_mask, &state})
            s->reset_data();
    }
    void save(const Operands& in, AttnProblem& problem, const AttnResult& r) {
        torch::autograd::set_history(r.out, getptr());
        packed = in.packed;
        for (int i = 0; i < (packed ? 1 : 3); ++i) x[i] = keep(in.t[i]);
        prepare = problem.prepared_from.defined();
        bias = keep(prepare ? problem.prepared_from : problem.bias);
        lse = keep(r.lse), keep_mask = keep(r.keep_mask);
        state = keep(problem.drop.state);
        out = keep(r.out, true);
        problem.bias = Tensor(), problem.prepared_from = Tensor(), problem.drop.state = Tensor();
        a = problem;
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list res(packed ? 1 : 3);
        if (!grads[0].defined()) return res;
        AttnProblem call = a;
        Operands in;
        Tensor dst[3];
        void* dst_ptr[3];
        int64_t ds[3][3];
        const Tensor tout = unpack_dense(out, getptr()), tlse = unpack_dense(lse);
        const c10::OptionalDeviceGuard guard(tout.device());
        if (packed) {
            in.take_packed(call, x[0].unpack());
            dst[0] = fresh_like(in.t[0]);
            Operands::packed_views<void>(call, mptr(dst[0]), dst_ptr, ds[0], ds[1], ds[2]);
        } else {
            in.take(call, x[0].unpack(), x[1].unpack(), x[2].unpack());
            for (int i = 0; i < 3; ++i) {
                dst[i] = fresh_like(in.t[i]);
                dst_ptr[i] = mptr(dst[i]);
                for (int j = 0; j < 3; ++j) ds[i][j] = dst[i].stride(j);
            }
        }
        if (call.empty() || call.sk() == 0) {
            for (const Tensor& t : dst)
                if (t.defined()) t.zero_();
        } else {
            if (prepare) {
                call.set_bias(bias.unpack(), false);
            } else {
                call.bias = bias.unpack();
                if (call.bias_type == SLAPO_BIAS_PREPARED)
                    call.bias = call.bias.contiguous();
                else if (call.bias.defined())
                    call.address_bias();
            }
            call.drop.state = unpack_dense(state);
            if (call.drop.state.defined())
                call.prm.plan.rng_state = call.drop.state.const_data_ptr();
            launch_attn_bwd(call, in, tout, tlse, unpack_dense(keep_mask), grads[0], dst_ptr, ds);
        }
        for (size_t i = 0; i < res.size(); ++i)
            if (task_should_compute_output(i)) res[i] = dst[i];
        return res;
    }
};

// What the two forms of the call share once the problem is described and the operands are taken.
AttnResult run_attention(AttnProblem& a, const Operands& x, at::IntArrayRef out_sizes,
                         const Tensor& mask, Dropout&& drop, bool need, bool save_mask,
                         int64_t save_mask_max) {
    a.set_bias(mask, !need && drop.p == 0.0);
    a.set_dropout(std::move(drop), x.t[0].device());
    // a mask geometry that the forward kernel would draw score by score is drawn ahead of it, which
    // takes the buffer also where no backward will read it
    const slapo_dropout_plan& plan = a.drop.plan;
    const bool per_score = a.drop.p > 0.0 &&
                           (plan.vec < 4 || a.sk() % 4 != 0 ||
                            (plan.total_threads & (plan.total_threads - 1)) != 0);
    return launch_attn_fwd(a, x, out_sizes, save_mask && a.drop.p < 1.0 && (need || per_score),
                           save_mask_max);
}

Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask_in,
                 bool causal, int64_t window, std::optional<double> scale, Dropout&& drop,
                 bool save_mask, int64_t save_mask_max) {
    check_operands(q, k, v);
    require_device({&mask_in});
    const Tensor mask = detached(mask_in);
    refuse_tangents({&q, &k, &v});
    const bool need = torch::autograd::compute_requires_grad(q, k, v);
    auto node = make_node<AttnBackward>(need, q, k, v);
    AttnProblem a;
    AttnResult r;
    Operands x;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(q.device());
        a.describe(q.scalar_type(), q.size(0), q.size(1), k.size(1), q.size(2), q.size(3), causal,
                   window, scale);
        x.take(a, q, k, v);
        r = run_attention(a, x, {a.b(), a.sq(), a.h(), a.d()}, mask, std::move(drop), need,
                          save_mask, save_mask_max);
    }
    if (node) node->save(x, a, r);
    return r.out;
}

// Self-attention on the output of a fused projection: qkv is [B, S, heads * 3 * head_dim] with q, k, v
// of one head side by side, the result [B, S, heads * head_dim].
Tensor attention_packed(const Tensor& qkv, int64_t head_dim, const Tensor& mask_in, bool causal,
                        int64_t window, std::optional<double> scale, Dropout&& drop, bool save_mask,
                        int64_t save_mask_max) {
    require_device({&qkv, &mask_in});
    const Tensor mask = detached(mask_in);
    refuse_tangents({&qkv});
    check_packed(qkv, head_dim);
    const bool need = torch::autograd::compute_requires_grad(qkv);
    auto node = make_node<AttnBackward>(need, qkv);
    AttnProblem a;
    AttnResult r;
    Operands x;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(qkv.device());
        a.describe(qkv.scalar_type(), qkv.size(0), qkv.size(1), qkv.size(1),
                   qkv.size(2) / (3 * head_dim), head_dim, causal, window, scale);
        x.take_packed(a, qkv);
        r = run_attention(a, x, {a.b(), a.sq(), a.h() * a.d()}, mask, std::move(drop), need,
                          save_mask, save_mask_max);
    }
    if (node) node->save(x, a, r);
    return r.out;
}

// ---- FusedQKV -----------------------------------------------------------------------------------

struct QkvSplitBackward : Node {
    std::vector<int64_t> sizes;  // of the packed tensor
    at::ScalarType dtype = at::kFloat;
    c10::Device device = at::kCPU;

    std::string name() const override { return "HipQKVSplitBackward"; }
    variable_list apply(variable_list&& grads) override {
        variable_list res(1);
        if (!grads[0].defined() && !grads[1].defined() && !grads[2].defined()) return res;
        const c10::OptionalDeviceGuard guard(device);
        if (c10::GradMode::is_enabled()) {  // create_graph: of operations that can be derived again
            Tensor like;
            for (const Tensor& t : grads)
                if (t.defined()) like = t;
            std::vector<Tensor> parts;
            for (const Tensor& t : grads) parts.push_back(t.defined() ? t : at::zeros_like(like));
            res[0] = at::stack(parts, -1).reshape(sizes);
            return res;
        }
        Tensor g[3];
        const Tensor packed = fresh(sizes, dtype);
        for (int i = 0; i < 3; ++i) {
            if (grads[i].defined())
                g[i] = dense(grads[i], dtype);
            else
                g[i] = fresh({packed.numel() / 3}, dtype).zero_();
        }
        if (packed.numel() > 0)
            check(slapo_amd_qkv_join(cptr(g[0]), cptr(g[1]), cptr(g[2]), mptr(packed),
                                     packed.numel() / 3, dtype_code(dtype), stream_of(packed)),
                  "slapo_amd_qkv_join");
        res[0] = packed;
        return res;
    }
};

// Whether qkv_split stands in for the torch operations: not where something watches those (vmap and
// the other function transforms, forward-mode differentiation, tracing, a dispatch mode) and not for
// types that the kernel does not move.
bool qkv_plain(const Tensor& packed) {
    const auto t = packed.scalar_type();
    return packed.is_cuda() && (t == at::kFloat || t == at::kHalf || t == at::kBFloat16) &&
           !packed.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched,
                                                          c10::DispatchKey::FuncTorchGradWrapper,
                                                          c10::DispatchKey::Functionalize,
                                                          c10::DispatchKey::Python})) &&
           !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !torch::jit::tracer::isTracing() && !packed._fw_grad(0).defined();
}

// [.., heads * head_size * 3] -> three [.., heads, head_size]
std::array<Tensor, 3> qkv_split(const Tensor& packed_in, int64_t heads, int64_t head_size) {
    require_device({&packed_in});
    refuse_tangents({&packed_in});
    TORCH_CHECK(packed_in.dim() > 0 && packed_in.size(-1) == heads * head_size * 3,
                "expected ", heads * head_size * 3, " columns, got ", packed_in.sizes());
    auto node = make_node<QkvSplitBackward>(torch::autograd::compute_requires_grad(packed_in),
                                            packed_in);
    std::array<Tensor, 3> out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(packed_in.device());
        const Tensor packed = packed_in.contiguous();
        const int code = dtype_code(packed.scalar_type());
        std::vector<int64_t> sizes(packed.sizes().begin(), packed.sizes().end() - 1);
        sizes.push_back(heads), sizes.push_back(head_size);
        for (Tensor& t : out) t = fresh(sizes, packed.scalar_type());
        if (packed.numel() > 0)
            check(slapo_amd_qkv_split(cptr(packed), mptr(out[0]), mptr(out[1]), mptr(out[2]),
                                      packed.numel() / 3, code, stream_of(packed)),
                  "slapo_amd_qkv_split");
    }
    if (node) {
        node->sizes.assign(packed_in.sizes().begin(), packed_in.sizes().end());
        node->dtype = packed_in.scalar_type();
        node->device = packed_in.device();
        for (const Tensor& t : out) torch::autograd::set_history(t, node);
    }
    return out;
}

// ---- cross entropy ------------------------------------------------------------------------------

struct CrossEntropyBackward : Node {
    SavedVariable logits, target, stats;  // stats: row maximum and 1 / sum, [2, rows]
    double smoothing = 0.0;

    std::string name() const override { return "HipCrossEntropyBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* s : {&logits, &target, &stats}) s->reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list res(1);
        if (!grads[0].defined()) return res;
        const Tensor x = unpack_dense(logits), t = unpack_dense(target), st = unpack_dense(stats);
        const c10::OptionalDeviceGuard guard(x.device());
        const Tensor g = dense(grads[0], at::kFloat);
        res[0] = fresh_like(x);
        const int64_t rows = t.numel();
        if (x.numel() == 0) return res;
        const float* m = static_cast<const float*>(cptr(st));
        check(slapo_amd_vocab_ce_bwd(cptr(x), static_cast<const int64_t*>(cptr(t)), m, m + rows,
                                     static_cast<const float*>(cptr(g)), mptr(res[0]), rows,
                                     x.size(-1), 0, smoothing, dtype_code(x.scalar_type()),
                                     stream_of(x)),
              "slapo_amd_vocab_ce_bwd");
        return res;
    }
};

Tensor cross_entropy(const Tensor& logits_in, const Tensor& target_in, double smoothing) {
    require_device({&logits_in, &target_in});
    refuse_tangents({&logits_in});
    TORCH_CHECK_VALUE(logits_in.dim() > 0, "logits need a vocabulary dimension");
    const int64_t vocab = logits_in.size(-1), rows = vocab > 0 ? logits_in.numel() / vocab : 0;
    TORCH_CHECK_VALUE(target_in.numel() == rows,
                      "target must have the shape of the logits without the vocabulary dim");
    TORCH_CHECK_VALUE(smoothing == 0.0 || vocab >= 2, "label smoothing needs at least two classes");
    auto node = make_node<CrossEntropyBackward>(torch::autograd::compute_requires_grad(logits_in),
                                                logits_in);
    Tensor logits, target, loss, stats;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(logits_in.device());
        logits = logits_in.contiguous();
        target = dense(target_in, at::kLong);
        const int code = dtype_code(logits.scalar_type());
        loss = fresh(target_in.sizes(), at::kFloat);
        stats = floats(2 * rows);
        float* m = static_cast<float*>(mptr(stats));
        if (rows > 0)
            check(slapo_amd_vocab_ce_loss(cptr(logits), static_cast<const int64_t*>(cptr(target)),
                                          static_cast<float*>(mptr(loss)), m, m + rows, rows, vocab,
                                          smoothing, code, stream_of(logits)),
                  "slapo_amd_vocab_ce_loss");
    }
    if (node) {
        torch::autograd::set_history(loss, node);
        node->logits = keep(logits), node->target = keep(target), node->stats = keep(stats);
        node->smoothing = smoothing;
    }
    return loss;
}

// ---- bias + GeLU --------------------------------------------------------------------------------

// rows x cols of x, with a bias of shape [cols]
std::pair<int64_t, int64_t> rows_cols(const Tensor& x, const Tensor& bias) {
    TORCH_CHECK_VALUE(x.dim() > 0, "the input needs at least one dimension");
    const int64_t cols = x.size(-1);
    TORCH_CHECK_VALUE(!bias.defined() || (bias.dim() == 1 && bias.size(0) == cols),
                      "bias must have shape [", cols, "], got ", bias.sizes());
    return {cols > 0 ? x.numel() / cols : 0, cols};
}

Tensor colsum_workspace(int64_t rows, int64_t cols, size_t* bytes) {
    *bytes = slapo_amd_colsum_workspace_bytes(rows, cols);
    return floats((int64_t)(*bytes / 4));
}

struct BiasGeluBackward : Node {
    SavedVariable y, bias;
    at::ScalarType bias_dtype = at::kFloat;

    std::string name() const override { return "HipBiasGeLUBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        y.reset_data(), bias.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list res(2);
        if (!grads[0].defined()) return res;
        const bool need_bias = task_should_compute_output(1);
        const Tensor ty = unpack_dense(y), tb = unpack_dense(bias);
        const c10::OptionalDeviceGuard guard(ty.device());
        const Tensor g = dense(grads[0], ty.scalar_type());
        const auto [rows, cols] = rows_cols(ty, tb);
        Tensor dx = fresh_like(ty), db, ws;
        if (need_bias) db = fresh({cols}, ty.scalar_type());
        if (ty.numel() == 0) {
            if (need_bias) db.zero_();
        } else {
            size_t ws_bytes = 0;
            if (need_bias) ws = colsum_workspace(rows, cols, &ws_bytes);
            check(slapo_amd_bias_gelu_bwd(cptr(g), cptr(ty), cptr(tb), mptr(dx), mptr(db), mptr(ws),
                                          ws_bytes, rows, cols, dtype_code(ty.scalar_type()),
                                          stream_of(ty)),
                  "slapo_amd_bias_gelu_bwd");
        }
        if (task_should_compute_output(0)) res[0] = dx;
        if (need_bias) res[1] = cast(db, bias_dtype);
        return res;
    }
};

// gelu_tanh(inp + bias); without a bias (an undefined tensor) a row of zeros stands in
Tensor bias_gelu(const Tensor& inp, const Tensor& bias_in) {
    require_device({&inp, &bias_in});
    refuse_tangents({&inp, &bias_in});
    auto node = make_node<BiasGeluBackward>(
        torch::autograd::compute_requires_grad(inp, bias_in), inp, bias_in);
    Tensor y, bias, out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(inp.device());
        const auto [rows, cols] = rows_cols(inp, bias_in);
        y = inp.contiguous();
        bias = bias_in.defined() ? dense(bias_in, y.scalar_type()) : at::zeros({cols}, y.options());
        out = fresh_like(y);
        const int code = dtype_code(y.scalar_type());
        if (y.numel() != 0)
            check(slapo_amd_bias_gelu_fwd(cptr(y), cptr(bias), mptr(out), rows, cols, code,
                                          stream_of(y)),
                  "slapo_amd_bias_gelu_fwd");
    }
    if (node) {
        torch::autograd::set_history(out, node);
        node->y = keep(y), node->bias = keep(bias);
        node->bias_dtype = bias_in.defined() ? bias_in.scalar_type() : y.scalar_type();
    }
    return out;
}

// ---- bias + dropout (+ residual) ----------------------------------------------------------------

struct BiasDropoutBackward : Node {
    Dropout drop;
    SavedVariable state;
    at::ScalarType bias_dtype = at::kFloat;
    bool has_residual = false;

    std::string name() const override { return "HipBiasDropoutResidualBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        state.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list res(3);
        if (!grads[0].defined()) return res;
        const bool need_x = task_should_compute_output(0), need_bias = task_should_compute_output(1);
        if (has_residual && task_should_compute_output(2)) res[2] = grads[0];
        // without dropout the gradient of x is the incoming one: only its column sum is left to do
        const bool pass_x = drop.p == 0.0;
        if (need_x && pass_x) res[0] = grads[0];
        const bool write_x = need_x && !pass_x;
        if (!write_x && !need_bias) return res;
        const c10::OptionalDeviceGuard guard(grads[0].device());
        const Tensor g = grads[0].contiguous();
        const auto [rows, cols] = rows_cols(g, Tensor());
        Tensor dx, db, ws;
        if (write_x) dx = fresh_like(g);
        if (need_bias) db = fresh({cols}, g.scalar_type());
        if (g.numel() == 0) {
            if (need_bias) db.zero_();
        } else {
            Dropout d = drop;
            d.state = unpack_dense(state);
            if (d.state.defined()) d.plan.rng_state = d.state.const_data_ptr();
            size_t ws_bytes = 0;
            if (need_bias) ws = colsum_workspace(rows, cols, &ws_bytes);
            check(slapo_amd_bias_dropout_residual_bwd(
                      cptr(g), mptr(dx), mptr(db), mptr(ws), ws_bytes, rows, cols,
                      dtype_code(g.scalar_type()), d.p, d.seed, d.offset, d.plan_ptr(),
                      stream_of(g)),
                  "slapo_amd_bias_dropout_residual_bwd");
        }
        if (write_x) res[0] = dx;
        if (need_bias) res[1] = cast(db, bias_dtype);
        return res;
    }
};

Tensor bias_dropout_residual(const Tensor& x_in, const Tensor& bias_in, const Tensor& res_in,
                             Dropout&& drop) {
    require_device({&x_in, &bias_in, &res_in});
    refuse_tangents({&x_in, &bias_in, &res_in});
    TORCH_CHECK_VALUE(!res_in.defined() || res_in.sizes() == x_in.sizes(),
                      "residual must have the shape of x");
    auto node = make_node<BiasDropoutBackward>(
        torch::autograd::compute_requires_grad(x_in, bias_in, res_in), x_in, bias_in, res_in);
    Tensor out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(x_in.device());
        const auto [rows, cols] = rows_cols(x_in, bias_in);
        const Tensor x = x_in.contiguous();
        const at::ScalarType dt = x.scalar_type();
        const Tensor bias = dense(bias_in, dt), res = dense(res_in, dt);
        const int code = dtype_code(dt);
        out = fresh_like(x);
        if (x.numel() == 0) drop.p = 0.0;
        drop.set_plan(x.numel(), (int)x.element_size(), x.device());
        if (x.numel() != 0)
            check(slapo_amd_bias_dropout_residual_fwd(
                      cptr(x), cptr(bias), cptr(res), mptr(out), rows, cols, code, drop.p,
                      drop.seed, drop.offset, drop.plan_ptr(), stream_of(x)),
                  "slapo_amd_bias_dropout_residual_fwd");
    }
    if (node) {
        torch::autograd::set_history(out, node);
        node->state = keep(drop.state);
        drop.state = Tensor();
        node->drop = drop;
        node->bias_dtype = bias_in.scalar_type();
        node->has_residual = res_in.defined();
    }
    return out;
}

// ---- bias + dropout + residual + LayerNorm ------------------------------------------------------

struct LayerNormBackward : Node {
    Dropout drop;
    SavedVariable z, stats, weight, state;  // stats: mean and rstd, [2, rows]
    at::ScalarType dtypes[3];               // bias, weight, ln_bias
    bool has_bias = false, has_residual = false;

    std::string name() const override { return "HipBiasDropoutResidualLayerNormBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* s : {&z, &stats, &weight, &state}) s->reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list res(5);  // x, bias, residual, weight, ln_bias
        if (!grads[0].defined()) return res;
        const Tensor tz = unpack_dense(z), tstats = unpack_dense(stats), tw = unpack_dense(weight);
        const c10::OptionalDeviceGuard guard(tz.device());
        const at::ScalarType dt = tz.scalar_type();
        const Tensor g = dense(grads[0], dt);
        const auto [rows, cols] = rows_cols(tz, Tensor());
        const bool need[5] = {task_should_compute_output(0),
                              has_bias && task_should_compute_output(1),
                              has_residual && task_should_compute_output(2),
                              task_should_compute_output(3), task_should_compute_output(4)};
        Tensor dx, dres, vec[3];  // vec: dbias, dweight, dln_bias
        // without dropout dx and dresidual are the same values: one tensor serves both
        const bool same = drop.p == 0.0 && need[0] && need[2];
        if (need[0]) dx = fresh_like(tz);
        if (need[2] && !same) dres = fresh_like(tz);
        const bool need_vec[3] = {need[1], need[3], need[4]};
        for (int i = 0; i < 3; ++i)
            if (need_vec[i]) vec[i] = fresh({cols}, tz.scalar_type());
        if (tz.numel() == 0) {
            for (Tensor& t : vec)
                if (t.defined()) t.zero_();
        } else if (need[0] || need[1] || need[2] || need[3] || need[4]) {
            Dropout d = drop;
            d.state = unpack_dense(state);
            if (d.state.defined()) d.plan.rng_state = d.state.const_data_ptr();
            Tensor ws;
            size_t ws_bytes = 0;
            if (need[1] || need[3] || need[4]) {
                ws_bytes = slapo_amd_ln_bwd_workspace_bytes(rows, cols);
                ws = floats((int64_t)(ws_bytes / 4));
            }
            const float* mean = static_cast<const float*>(cptr(tstats));
            check(slapo_amd_bias_dropout_residual_ln_bwd(
                      cptr(g), cptr(tz), mean, mean + rows, cptr(tw), mptr(dx), mptr(dres),
                      mptr(vec[1]), mptr(vec[2]), mptr(vec[0]), mptr(ws), ws_bytes, rows, cols,
                      dtype_code(dt), d.p, d.seed, d.offset, d.plan_ptr(), stream_of(tz)),
                  "slapo_amd_bias_dropout_residual_ln_bwd");
        }
        res[0] = dx;
        res[1] = cast(vec[0], dtypes[0]);
        res[2] = same ? dx : dres;
        res[3] = cast(vec[1], dtypes[1]);
        res[4] = cast(vec[2], dtypes[2]);
        return res;
    }
};

Tensor bias_dropout_residual_layer_norm(const Tensor& x_in, const Tensor& bias_in,
                                        const Tensor& res_in, const Tensor& weight_in,
                                        const Tensor& ln_bias_in, double eps, Dropout&& drop) {
    require_device({&x_in, &bias_in, &res_in, &weight_in, &ln_bias_in});
    refuse_tangents({&x_in, &bias_in, &res_in, &weight_in, &ln_bias_in});
    TORCH_CHECK_VALUE(!res_in.defined() || res_in.sizes() == x_in.sizes(),
                      "residual must have the shape of x");
    for (const Tensor* t : {&bias_in, &weight_in, &ln_bias_in})
        TORCH_CHECK_VALUE(
            !t->defined() || (t->dim() == 1 && x_in.dim() > 0 && t->size(0) == x_in.size(-1)),
            "bias, weight and ln_bias must be 1-D of the last dimension of x");
    const bool need = torch::autograd::compute_requires_grad(x_in, bias_in, res_in, weight_in,
                                                             ln_bias_in);
    auto node =
        make_node<LayerNormBackward>(need, x_in, bias_in, res_in, weight_in, ln_bias_in);
    Tensor y, z, stats, weight;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(x_in.device());
        const auto [rows, cols] = rows_cols(x_in, Tensor());
        const Tensor x = x_in.contiguous();
        const at::ScalarType dt = x.scalar_type();
        const Tensor bias = dense(bias_in, dt), res = dense(res_in, dt);
        weight = dense(weight_in, dt);
        const Tensor ln_bias = dense(ln_bias_in, dt);
        const int code = dtype_code(dt);
        y = fresh_like(x);
        if (need) {
            z = fresh_like(x);
            stats = floats(2 * rows);
        }
        if (x.numel() == 0) drop.p = 0.0;
        drop.set_plan(x.numel(), (int)x.element_size(), x.device());
        float* mean = static_cast<float*>(mptr(stats));
        if (x.numel() != 0)
            check(slapo_amd_bias_dropout_residual_ln_fwd(
                      cptr(x), cptr(bias), cptr(res), cptr(weight), cptr(ln_bias), mptr(z),
                      mptr(y), mean, mean ? mean + rows : nullptr, rows, cols, code, eps, drop.p,
                      drop.seed, drop.offset, drop.plan_ptr(), stream_of(x)),
                  "slapo_amd_bias_dropout_residual_ln_fwd");
    }
    if (node) {
        torch::autograd::set_history(y, node);
        node->z = keep(z), node->stats = keep(stats), node->weight = keep(weight);
        node->state = keep(drop.state);
        drop.state = Tensor();
        node->drop = drop;
        node->has_bias = bias_in.defined(), node->has_residual = res_in.defined();
        node->dtypes[0] = bias_in.defined() ? bias_in.scalar_type() : at::kFloat;
        node->dtypes[1] = weight_in.scalar_type();
        node->dtypes[2] = ln_bias_in.scalar_type();
    }
    return y;
}

// ---- random numbers -----------------------------------------------------------------------------

// (seed, offset) for one launch from the default generator of device `index`, whose offset moves
// on by `increment`, as an ATen random kernel would have it.
std::pair<uint64_t, uint64_t> draw(int64_t increment, c10::DeviceIndex index) {
    at::Generator gen = at::globalContext().defaultGenerator(at::Device(at::kCUDA, index));
    std::lock_guard<std::mutex> lock(gen.mutex());
    const uint64_t seed = gen.current_seed(), offset = gen.get_offset();
    gen.set_offset(offset + (uint64_t)increment);
    return {seed, offset};
}

// ---- Python -------------------------------------------------------------------------------------

const Tensor& tensor_arg(PyObject* o, const char* name) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), name, " must be a tensor, got ", Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}
const Tensor& optional_tensor_arg(PyObject* o, const char* name) {
    static const Tensor none;
    return o == Py_None ? none : tensor_arg(o, name);
}
double double_arg(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
}
int64_t int_arg(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}
uint64_t uint_arg(PyObject* o) {
    const unsigned long long v = PyLong_AsUnsignedLongLong(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) throw python_error();
    return v;
}
bool bool_arg(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw python_error();
    return v != 0;
}
// p, seed, offset, state
Dropout dropout_args(PyObject* const* a) {
    Dropout d;
    d.p = double_arg(a[0]);
    d.seed = uint_arg(a[1]);
    d.offset = uint_arg(a[2]);
    d.state = optional_tensor_arg(a[3], "rng_state");
    return d;
}
void want(Py_ssize_t n, Py_ssize_t expected, const char* name) {
    TORCH_CHECK_TYPE(n == expected, name, " takes ", expected, " arguments, got ", n);
}

// attention(q, k, v, mask, causal, window, scale, p, seed, offset, state, save_mask, save_max)
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 13, "attention");
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
    const Tensor& mask = optional_tensor_arg(a[3], "attention_mask");
    const bool causal = bool_arg(a[4]), save_mask = bool_arg(a[11]);
    const int64_t window = int_arg(a[5]), save_max = int_arg(a[12]);
    std::optional<double> scale;
    if (a[6] != Py_None) scale = double_arg(a[6]);
    Dropout drop = dropout_args(a + 7);
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = attention(q, k, v, mask, causal, window, scale, std::move(drop), save_mask, save_max);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// attention_packed(qkv, head_dim, mask, causal, window, scale, p, seed, offset, state, save_mask,
// save_max)
PyObject* py_attention_packed(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 12, "attention_packed");
    const Tensor& qkv = tensor_arg(a[0], "qkv");
    const int64_t head_dim = int_arg(a[1]);
    const Tensor& mask = optional_tensor_arg(a[2], "attention_mask");
    const bool causal = bool_arg(a[3]), save_mask = bool_arg(a[10]);
    const int64_t window = int_arg(a[4]), save_max = int_arg(a[11]);
    std::optional<double> scale;
    if (a[5] != Py_None) scale = double_arg(a[5]);
    Dropout drop = dropout_args(a + 6);
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = attention_packed(qkv, head_dim, mask, causal, window, scale, std::move(drop),
                               save_mask, save_max);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// qkv_plain(packed)
PyObject* py_qkv_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 1, "qkv_plain");
    return PyBool_FromLong(qkv_plain(tensor_arg(a[0], "packed")));
    END_HANDLE_TH_ERRORS
}

// qkv_split(packed, heads, head_size): [q, k, v]
PyObject* py_qkv_split(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 3, "qkv_split");
    const Tensor& packed = tensor_arg(a[0], "packed");
    const int64_t heads = int_arg(a[1]), head_size = int_arg(a[2]);
    std::array<Tensor, 3> out;
    {
        pybind11::gil_scoped_release no_gil;
        out = qkv_split(packed, heads, head_size);
    }
    THPObjectPtr list(PyList_New(3));
    if (!list) throw python_error();
    for (int i = 0; i < 3; ++i)
        PyList_SET_ITEM(list.get(), i, THPVariable_Wrap(std::move(out[i])));
    return list.release();
    END_HANDLE_TH_ERRORS
}

// cross_entropy(logits, target, smoothing)
PyObject* py_cross_entropy(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 3, "cross_entropy");
    const Tensor &logits = tensor_arg(a[0], "logits"), &target = tensor_arg(a[1], "target");
    const double smoothing = double_arg(a[2]);
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = cross_entropy(logits, target, smoothing);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// attention_scores(q, k, v, mask): checks the operands -- before anything is drawn for them -- and
// returns the number of scores B * H * Sq * Sk
PyObject* py_attention_scores(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 4, "attention_scores");
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
    check_operands(q, k, v);
    check_mask(optional_tensor_arg(a[3], "attention_mask"),
               {q.size(0), q.size(2), q.size(1), k.size(1)});
    return PyLong_FromLongLong(q.size(0) * q.size(1) * q.size(2) * k.size(1));
    END_HANDLE_TH_ERRORS
}

// packed_scores(qkv, head_dim, mask): the same for the packed form
PyObject* py_packed_scores(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 3, "packed_scores");
    const Tensor& qkv = tensor_arg(a[0], "qkv");
    const int64_t head_dim = int_arg(a[1]);
    check_packed(qkv, head_dim);
    const int64_t b = qkv.size(0), s = qkv.size(1), h = qkv.size(2) / (3 * head_dim);
    check_mask(optional_tensor_arg(a[2], "attention_mask"), {b, h, s, s});
    return PyLong_FromLongLong(b * h * s * s);
    END_HANDLE_TH_ERRORS
}

PyObject* py_bias_gelu(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 2, "bias_gelu");
    const Tensor& x = tensor_arg(a[0], "inp");
    const Tensor& bias = optional_tensor_arg(a[1], "bias");
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = bias_gelu(x, bias);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// bias_dropout_residual(x, bias, residual, p, seed, offset, state)
PyObject* py_bias_dropout_residual(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 7, "bias_dropout_residual");
    const Tensor &x = tensor_arg(a[0], "x"), &bias = tensor_arg(a[1], "bias");
    const Tensor& residual = optional_tensor_arg(a[2], "residual");
    Dropout drop = dropout_args(a + 3);
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = bias_dropout_residual(x, bias, residual, std::move(drop));
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// bias_dropout_residual_layer_norm(x, bias, residual, weight, ln_bias, eps, p, seed, offset, state)
PyObject* py_layer_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 10, "bias_dropout_residual_layer_norm");
    const Tensor& x = tensor_arg(a[0], "x");
    const Tensor& bias = optional_tensor_arg(a[1], "bias");
    const Tensor& residual = optional_tensor_arg(a[2], "residual");
    const Tensor &weight = tensor_arg(a[3], "weight"), &ln_bias = tensor_arg(a[4], "ln_bias");
    const double eps = double_arg(a[5]);
    Dropout drop = dropout_args(a + 6);
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = bias_dropout_residual_layer_norm(x, bias, residual, weight, ln_bias, eps,
                                               std::move(drop));
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// philox_increment(numel, elem_bytes, device_index): how far F.dropout would advance the generator
PyObject* py_philox_increment(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 3, "philox_increment");
    slapo_dropout_plan plan;
    check(slapo_amd_dropout_plan(int_arg(a[0]), (int)int_arg(a[1]), 256, (int)int_arg(a[2]), &plan),
          "slapo_amd_dropout_plan");
    return PyLong_FromLongLong(plan.offset_increment);
    END_HANDLE_TH_ERRORS
}

// draw(increment, device_index): (seed, offset), or None while the current stream is capturing
PyObject* py_draw(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    want(n, 2, "draw");
    const int64_t increment = int_arg(a[0]), index = int_arg(a[1]);
    if (capturing()) Py_RETURN_NONE;
    const auto [seed, offset] = draw(increment, (c10::DeviceIndex)index);
    return Py_BuildValue("KK", (unsigned long long)seed, (unsigned long long)offset);
    END_HANDLE_TH_ERRORS
}

#define SLAPO_METHOD(name, fn) \
    { name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr }
PyMethodDef methods[] = {
    SLAPO_METHOD("attention", py_attention),
    SLAPO_METHOD("attention_packed", py_attention_packed),
    SLAPO_METHOD("attention_scores", py_attention_scores),
    SLAPO_METHOD("packed_scores", py_packed_scores),
    SLAPO_METHOD("qkv_plain", py_qkv_plain),
    SLAPO_METHOD("qkv_split", py_qkv_split),
    SLAPO_METHOD("cross_entropy", py_cross_entropy),
    SLAPO_METHOD("bias_gelu", py_bias_gelu),
    SLAPO_METHOD("bias_dropout_residual", py_bias_dropout_residual),
    SLAPO_METHOD("bias_dropout_residual_layer_norm", py_layer_norm),
    SLAPO_METHOD("philox_increment", py_philox_increment),
    SLAPO_METHOD("draw", py_draw),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host",
                          "Native host path of the slapo_amd ops", -1, methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module_def); }
