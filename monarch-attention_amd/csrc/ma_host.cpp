// Host side of the "hip" implementation: from torch tensors to the C ABI of libma_hip.so (include/ma_hip.h), with the
// autograd node of a training step.  A Python extension module; ma/ma_hip.py holds the functions that call it and the
// texts of the argument errors.
//
// A small forward takes 3 - 10 us on the GPU, and the calls of a training step of a short sequence take 40 us, so the host
// path is what such callers wait for: with the parameter blocks filled from Python, through ctypes and
// torch.autograd.Function, a forward call took 8 - 11 us of host time and a training step 190 - 230 us whatever its size.
// Here a forward call costs an allocation, a launch and about a microsecond of Python.
//
// The library is bound by path (bind()), not linked: MA_HIP_LIBRARY may name another build of it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <dlfcn.h>

#include <initializer_list>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/DeviceGuard.h>
#include <c10/core/AutogradState.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include "ma_hip.h"

namespace {

using at::Tensor;

// ---- the library
struct Api {
    const char* (*strerror)(int);
    int (*layout)(const ma_fwd_params*, ma_ws_layout*);
    uint64_t (*workspace_bytes)(const ma_fwd_params*);
    int (*fwd)(const ma_fwd_params*, void*);
    uint64_t (*state_bytes)(const ma_fwd_params*);
    uint64_t (*keep_workspace_bytes)(const ma_fwd_params*);
    int (*fwd_keep)(const ma_fwd_params*, void*, uint64_t, void*);
    uint64_t (*matrix_workspace_bytes)(const ma_fwd_params*);
    int (*matrix)(const ma_fwd_params*, float*, void*);
    uint64_t (*bwd_workspace_bytes)(const ma_bwd_params*);
    int (*bwd)(const ma_bwd_params*, void*);
    uint64_t (*bwd_kept_workspace_bytes)(const ma_bwd_params*);
    int (*bwd_kept)(const ma_bwd_params*, const void*, uint64_t, void*);
} api;

// ma/_hip_lib.py check(): the exception a non-zero status stands for
void check(int status, const char* what) {
    if (status == MA_OK) return;
    const std::string msg = std::string(what) + ": " + api.strerror(status) + " (status " + std::to_string(status) + ")";
    switch (status) {
        case MA_ERR_SHAPE: case MA_ERR_DTYPE: case MA_ERR_STRIDE: case MA_ERR_VARIANT: case MA_ERR_NULL: TORCH_CHECK_VALUE(false, msg);
        case MA_ERR_UNSUPPORTED: TORCH_CHECK_NOT_IMPLEMENTED(false, msg);
        default: TORCH_CHECK(false, msg);
    }
}

// ---- workspaces: one per (device, stream), grown on demand and reused call after call (calls on one stream are ordered,
// so they can share it).  Allocated zero-filled; every forward call leaves the sync area ready for the next one
// (MA_FLAG_SYNC_READY).  A one-launch kernel whose bounded wait runs out stores the code of the error into a word of
// pinned host memory, and EVERY call on the workspace looks at that word first (a plain host read).
// Calls run without the GIL.  `lock` is held over a call's launches: those of two threads on one stream must not
// interleave, they share the state arrays.
struct Workspace {
    std::mutex lock;
    Tensor buf, err_host;
    volatile int32_t* err = nullptr;
    bool dirty = false;   // a failed call: the sync area must be cleared before the next one

    void resize(c10::Device device, uint64_t nbytes) {
        // calls on this stream that still use the old buffer are ahead of everything queued from here on, and the
        // caching allocator hands a freed block to other streams only after that work is done
        buf = at::zeros({static_cast<int64_t>(std::max<uint64_t>(nbytes, 1u << 20))}, at::TensorOptions().dtype(at::kByte).device(device));
    }
    // lock held: the buffer has nbytes, and no earlier call on it failed
    void ready(c10::Device device, uint64_t nbytes) {
        if (err == nullptr) {
            err_host = at::zeros({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
            err = err_host.data_ptr<int32_t>();
        }
        if (!buf.defined() || static_cast<uint64_t>(buf.numel()) < nbytes) resize(device, nbytes);
        report();
    }
    void report() {
        if (err == nullptr || *err == 0) return;
        const int code = *err;
        *err = 0;
        dirty = true;
        buf.slice(0, 4, 8).zero_();   // the word in the workspace is sticky: clear it for the calls to come
        const std::string why = code == 1 ? "a bounded wait between workgroups ran out"
                                : code == 2 ? "workgroups of one head ran on different XCDs (the one-launch kernels rely on ids x, x + 8, ... "
                                              "sharing an XCD)"
                                            : "error word " + std::to_string(code);
        TORCH_CHECK(false, "monarch_attention_hip: an earlier forward call on this stream failed: ", why,
                    "; its output holds NaN rows.  The workspace has been reset; pass variant='staged' to avoid the one-launch kernels");
    }
};
std::mutex g_mutex;   // the map
std::map<std::pair<int, void*>, std::shared_ptr<Workspace>> g_workspaces;

std::shared_ptr<Workspace> workspace_of(c10::Device device, void* stream) {
    const std::lock_guard<std::mutex> lock(g_mutex);
    auto& w = g_workspaces[{device.index(), stream}];
    if (!w) w = std::make_shared<Workspace>();
    return w;
}

// The GIL is released while a call allocates and launches: a full queue blocks the launch.  Nothing that holds one of the
// locks above waits for them with the GIL.
struct NoGil {
    PyThreadState* const state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// ---- arguments
int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return MA_F32;
        case at::kHalf: return MA_F16;
        case at::kBFloat16: return MA_BF16;
        default: return -1;
    }
}

// the mask as the library reads it, in place, whatever its element type (non-zero = keep, ma/ma_torch.py:98)
int mask_code(at::ScalarType t) {
    switch (t) {
        case at::kBool: case at::kByte: case at::kChar: return MA_MASK_U8;
        case at::kShort: return MA_MASK_I16;
        case at::kInt: return MA_MASK_I32;
        case at::kLong: return MA_MASK_I64;
        case at::kHalf: return MA_MASK_F16;
        case at::kBFloat16: return MA_MASK_BF16;
        case at::kFloat: return MA_MASK_F32;
        case at::kDouble: return MA_MASK_F64;
        default: return -1;
    }
}

// Arguments of one operator call.  `mask` may be undefined.
struct Call {
    Tensor q, k, v, mask;
    int T, B, variant, flags;
    bool pre_pad;
};

// Is this a call the library can be asked to run?  (ma_hip._check_inputs says what is wrong with the others.)
bool valid(const Call& c) {
    const Tensor &q = c.q, &k = c.k, &v = c.v;
    if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
    const auto qs = q.sizes(), vs = v.sizes();
    if (qs != k.sizes() || vs[0] != qs[0] || vs[1] != qs[1] || vs[2] != qs[2]) return false;
    if (q.scalar_type() != k.scalar_type() || dtype_code(q.scalar_type()) < 0 || dtype_code(v.scalar_type()) < 0) return false;
    if (!q.is_cuda() || q.device() != k.device() || q.device() != v.device()) return false;
    if (q.numel() < 1 || v.numel() < 1 || c.T < 1 || c.B < 1) return false;
    if (c.mask.defined())
        if (c.mask.dim() != 2 || c.mask.size(0) != qs[0] || c.mask.size(1) != qs[2] || c.mask.device() != q.device() ||
            mask_code(c.mask.scalar_type()) < 0)
            return false;
    return true;
}

// Forward-mode AD: the operator has no jvp, and a result without a tangent would pass for a zero derivative.
void refuse_tangents(std::initializer_list<const Tensor*> tensors) {
    // (outside of every dual level - one lookup - there are none, and the tensors' metadata is not touched)
    if (!c10::AutogradState::get_tls_state().get_fw_grad_mode() || !torch::autograd::ForwardADLevel::try_get_by_idx(0)) return;
    for (const Tensor* t : tensors)
        TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(/*level=*/0).defined(),
                                    "monarch_attention_hip has no forward-mode derivative (jvp): q, k, v and the output gradient must not be dual tensors");
}

// The library wants unit stride along the last dimension and token rows that do not overlap; batch and head dimensions
// may be broadcast.  Anything else - e.g. an expand() along the tokens - is copied once.
Tensor rows_contiguous(const Tensor& t) {
    const auto size = t.sizes(), stride = t.strides();
    if ((stride[3] != 1 && size[3] != 1) || (size[2] > 1 && stride[2] < size[3])) return t.contiguous();
    return t;
}

void set_strides(int64_t (&dst)[3], const Tensor& t) {
    const auto s = t.strides();
    for (int i = 0; i < 3; ++i) dst[i] = s[i];
}

// q, k, v have rows_contiguous() layouts
ma_fwd_params params_of(const Call& c, const Tensor& q, const Tensor& k, const Tensor& v) {
    ma_fwd_params p = {};
    p.q = q.data_ptr();
    p.k = k.data_ptr();
    p.v = v.data_ptr();
    const auto size = q.sizes();
    p.E = static_cast<int32_t>(size[0]);
    p.H = static_cast<int32_t>(size[1]);
    p.N = static_cast<int32_t>(size[2]);
    p.D = static_cast<int32_t>(size[3]);
    p.Dv = static_cast<int32_t>(v.size(3));
    p.B = c.B;
    p.T = c.T;
    p.pre_pad = c.pre_pad;
    p.dtype_qk = dtype_code(q.scalar_type());
    p.dtype_v = dtype_code(v.scalar_type());
    p.variant = c.variant;
    p.flags = c.flags;
    set_strides(p.q_stride, q);
    set_strides(p.k_stride, k);
    set_strides(p.v_stride, v);
    if (c.mask.defined()) {
        p.mask = c.mask.data_ptr();
        p.mask_dtype = mask_code(c.mask.scalar_type());
        p.mask_stride[0] = c.mask.stride(0);
        p.mask_stride[1] = c.mask.stride(1);
    }
    p.eps = 1e-12f;   // ma/ma_torch.py:10,38
    return p;
}

// Output buffer in v's memory layout: models pass (E,H,N,D) views of (E,N,H,D) projections (experiments/vit/model.py:73-79)
// and turn the result back with permute(0, 2, 1, 3).contiguous() (:99) - with the output laid out likewise that copy is a
// no-op.  Anything else gets a contiguous (E,H,N,Dv) tensor.
Tensor output_like(const Tensor& v) {
    const auto n = v.sizes(), s = v.strides();
    const int64_t H = n[1], N = n[2], D = n[3];
    const bool tokens_first = H > 1 && N > 1 && (D == 1 || s[3] == 1) && s[1] == D && s[2] == H * D && (n[0] == 1 || s[0] == N * H * D);
    if (tokens_first && !v.is_contiguous()) return at::empty_strided(n, {N * H * D, D, H * D, 1}, v.options());
    return at::empty(n, v.options());
}

void* current_stream(c10::Device device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

Tensor device_bytes(uint64_t nbytes, const Tensor& like) {
    return at::empty({static_cast<int64_t>(nbytes)}, at::TensorOptions().dtype(at::kByte).device(like.device()));
}

// The forward call.  keep: also fill *state for the backward pass.
Tensor run_forward(const Call& c, Tensor* state) {
    const at::DeviceGuard guard(c.q.device());
    const Tensor q = rows_contiguous(c.q), k = rows_contiguous(c.k), v = rows_contiguous(c.v);
    Tensor out = output_like(v);
    ma_fwd_params p = params_of(c, q, k, v);
    p.out = out.data_ptr();
    set_strides(p.out_stride, out);
    const uint64_t nbytes = state ? api.keep_workspace_bytes(&p) : api.workspace_bytes(&p);
    if (nbytes == 0) {   // invalid problem: let the library say why
        ma_ws_layout unused;
        check(api.layout(&p, &unused), "monarch_attention_hip");
    }
    void* stream = current_stream(q.device());
    const std::shared_ptr<Workspace> w = workspace_of(q.device(), stream);
    const std::lock_guard<std::mutex> lock(w->lock);
    w->ready(q.device(), nbytes);
    p.workspace = w->buf.data_ptr();
    p.workspace_bytes = static_cast<uint64_t>(w->buf.numel());
    p.error_word = reinterpret_cast<uint32_t*>(const_cast<int32_t*>(w->err));
    if (w->dirty) {
        w->buf.zero_();
        w->dirty = false;
    }
    p.flags |= MA_FLAG_SYNC_READY;
    if (state) {
        *state = device_bytes(api.state_bytes(&p), q);
        check(api.fwd_keep(&p, state->data_ptr(), static_cast<uint64_t>(state->numel()), stream), "ma_fwd_keep");
    } else {
        check(api.fwd(&p, stream), "ma_fwd");
    }
    return out;
}

// The dense matrix (c.v unused)
Tensor run_matrix(const Call& c) {
    const c10::AutoGradMode no_grad(false);
    const at::DeviceGuard guard(c.q.device());
    const Tensor q = rows_contiguous(c.q), k = rows_contiguous(c.k);
    ma_fwd_params p = params_of(c, q, k, q);
    const int64_t N = q.size(2);
    const Tensor A = at::empty({q.size(0), q.size(1), N, N}, q.options().dtype(at::kFloat));
    p.out = A.data_ptr();
    set_strides(p.out_stride, q);
    if (p.E > 1 && p.out_stride[0] == 0) p.out_stride[0] = 1;   // stand-ins: the call reads neither out nor its strides
    if (p.H > 1 && p.out_stride[1] == 0) p.out_stride[1] = 1;
    const uint64_t nbytes = api.matrix_workspace_bytes(&p);
    if (nbytes == 0) {
        ma_ws_layout unused;
        check(api.layout(&p, &unused), "monarch_matrix_hip");
    }
    void* stream = current_stream(q.device());
    {
        const std::shared_ptr<Workspace> w = workspace_of(q.device(), stream);
        const std::lock_guard<std::mutex> lock(w->lock);
        w->report();
    }
    const Tensor ws = device_bytes(nbytes, q);   // (with the probabilities: allocated per call and freed after it)
    p.workspace = ws.data_ptr();
    p.workspace_bytes = nbytes;
    check(api.matrix(&p, A.data_ptr<float>(), stream), "ma_matrix");
    return A;
}

struct Grads {
    Tensor dq, dk, dv;
};

// The backward pass; state: what run_forward kept, or undefined.
Grads run_backward(const Call& c, const Tensor& dout_, const Tensor& state) {
    const at::DeviceGuard guard(c.q.device());
    const Tensor q = rows_contiguous(c.q), k = rows_contiguous(c.k), v = rows_contiguous(c.v);
    const Tensor dout = rows_contiguous(dout_.scalar_type() == v.scalar_type() ? dout_ : dout_.to(v.scalar_type()));
    Grads g{at::empty_like(q), at::empty_like(k), at::empty_like(v)};
    ma_bwd_params b = {};
    b.fwd = params_of(c, q, k, v);
    b.fwd.out = g.dv.data_ptr();   // not written
    set_strides(b.fwd.out_stride, g.dv);
    b.dout = dout.data_ptr();
    b.dq = g.dq.data_ptr();
    b.dk = g.dk.data_ptr();
    b.dv = g.dv.data_ptr();
    set_strides(b.dout_stride, dout);
    set_strides(b.dq_stride, g.dq);
    set_strides(b.dk_stride, g.dk);
    set_strides(b.dv_stride, g.dv);
    const uint64_t nbytes = state.defined() ? api.bwd_kept_workspace_bytes(&b) : api.bwd_workspace_bytes(&b);
    if (nbytes == 0) {
        ma_ws_layout unused;
        check(api.layout(&b.fwd, &unused), "monarch_attention_hip_backward");
        TORCH_CHECK_NOT_IMPLEMENTED(false, "ma_bwd does not support this problem (variant or block shape)");
    }
    const Tensor ws = device_bytes(nbytes, q);   // the gradients of every state: allocated per call and freed after it
    b.fwd.workspace = ws.data_ptr();
    b.fwd.workspace_bytes = nbytes;
    void* stream = current_stream(q.device());
    if (state.defined()) check(api.bwd_kept(&b, state.data_ptr(), static_cast<uint64_t>(state.numel()), stream), "ma_bwd_kept");
    else check(api.bwd(&b, stream), "ma_bwd");
    return g;
}

// One autograd node per operator call: forward ma_fwd_keep, backward ma_bwd_kept.  A forward variant that keeps no state
// in memory (an explicit 'fused' or 'resident') runs as ma_fwd, and ma_bwd runs the steps again.
struct MonarchAttentionHipBackward : public torch::autograd::Node {
    // the state goes through saved-tensor hooks as the inputs do: checkpointing drops it, save_on_cpu moves it
    torch::autograd::SavedVariable q, k, v, mask, state;
    bool has_mask = false, has_state = false;
    int64_t state_bytes = 0;
    Call call;   // without tensors

    std::string name() const override { return "MonarchAttentionHipBackward"; }

    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        q.reset_data();
        k.reset_data();
        v.reset_data();
        mask.reset_data();
        state.reset_data();
    }

    torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        torch::autograd::variable_list out(3);
        if (!grads[0].defined()) return out;
        refuse_tangents({&grads[0]});
        Call c = call;
        c.q = q.unpack();
        c.k = k.unpack();
        c.v = v.unpack();
        if (has_mask) c.mask = mask.unpack();
        Tensor st;
        if (has_state) st = state.unpack();
        Grads g;
        {
            const c10::AutoGradMode no_grad(false);
            if (has_state) {   // a hook may have put it anywhere
                TORCH_CHECK(st.defined() && st.scalar_type() == at::kByte && st.numel() == state_bytes && st.device() == c.q.device(),
                            "the kept state of monarch_attention_hip came back from its saved-tensor hooks as another tensor: expected ", state_bytes,
                            " bytes (uint8) on ", c.q.device());
                if (!st.is_contiguous() || reinterpret_cast<uintptr_t>(st.data_ptr()) % 256 != 0) st = st.clone(at::MemoryFormat::Contiguous);
            }
            g = run_backward(c, grads[0], st);
        }
        if (task_should_compute_output(0)) out[0] = std::move(g.dq);
        if (task_should_compute_output(1)) out[1] = std::move(g.dk);
        if (task_should_compute_output(2)) out[2] = std::move(g.dv);
        if (c10::GradMode::is_enabled() && grads[0].requires_grad()) {   // create_graph: there is no second derivative
            for (auto& t : out)
                if (t.defined()) t.set_requires_grad(true);
            torch::autograd::DelayedError error("trying to differentiate twice a function that was marked with @once_differentiable", 3);
            return error.apply(std::move(out));
        }
        return out;
    }
};

// keep: keep the state of the steps (the forward runs as a variant that has it in memory); else ma_fwd, and the backward
// runs the steps again.
Tensor run_recorded(const Call& c, bool keep) {
    auto node = std::shared_ptr<MonarchAttentionHipBackward>(new MonarchAttentionHipBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(c.q, c.k, c.v));
    const bool keeps = keep && c.variant != MA_VARIANT_FUSED && c.variant != MA_VARIANT_RESIDENT && c.variant != MA_VARIANT_SLICED;
    Tensor out, state;
    {
        const c10::AutoGradMode no_grad(false);
        out = run_forward(c, keeps ? &state : nullptr);
    }
    node->q = torch::autograd::SavedVariable(c.q, false);
    node->k = torch::autograd::SavedVariable(c.k, false);
    node->v = torch::autograd::SavedVariable(c.v, false);
    node->has_mask = c.mask.defined();
    if (node->has_mask) node->mask = torch::autograd::SavedVariable(c.mask, false);
    node->has_state = keeps;
    if (keeps) {
        node->state_bytes = state.numel();
        node->state = torch::autograd::SavedVariable(state, false);
    }
    node->call.T = c.T;
    node->call.B = c.B;
    node->call.pre_pad = c.pre_pad;
    // the backward kernels follow 'generic' and 'staged'; with any other variant they are chosen by the library
    node->call.variant = c.variant == MA_VARIANT_GENERIC || c.variant == MA_VARIANT_STAGED ? c.variant : MA_VARIANT_AUTO;
    node->call.flags = 0;
    torch::autograd::set_history(out, node);
    return out;
}

// ---- Python functions
// Fills T, B, pre_pad, variant, flags from args[0 .. 4]; false: not ints (the caller reports it)
bool scalars(PyObject* const* args, Call* c) {
    if (!PyLong_Check(args[0]) || !PyLong_Check(args[1])) return false;
    int overflow = 0;
    const long long T = PyLong_AsLongLongAndOverflow(args[0], &overflow);
    if (overflow || T < 1 || T > 0x7fffffff) return false;
    const long long B = PyLong_AsLongLongAndOverflow(args[1], &overflow);
    if (overflow || B < 1 || B > 0x7fffffff) return false;
    const int pre = PyObject_IsTrue(args[2]);
    if (pre < 0) throw python_error();
    c->T = static_cast<int>(T);
    c->B = static_cast<int>(B);
    c->pre_pad = pre != 0;
    c->variant = static_cast<int>(PyLong_AsLong(args[3]));
    c->flags = static_cast<int>(PyLong_AsLong(args[4]));
    return true;
}

bool tensor(PyObject* o, Tensor* t) {
    if (!THPVariable_Check(o)) return false;
    *t = THPVariable_Unpack(o);
    return true;
}

bool tensor_or_none(PyObject* o, Tensor* t) { return o == Py_None || tensor(o, t); }

// forward(q, k, v, mask, T, B, pre_pad, variant, flags, keep_state) -> Tensor, or None for arguments the operator does not take
PyObject* py_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    if (n != 10 || !tensor(args[0], &c.q) || !tensor(args[1], &c.k) || !tensor(args[2], &c.v)) Py_RETURN_NONE;
    refuse_tangents({&c.q, &c.k, &c.v});
    if (!tensor_or_none(args[3], &c.mask) || !scalars(args + 4, &c) || !valid(c)) Py_RETURN_NONE;
    const bool record = c10::GradMode::is_enabled() && (c.q.requires_grad() || c.k.requires_grad() || c.v.requires_grad());
    const int keep = PyObject_IsTrue(args[9]);
    if (keep < 0) throw python_error();
    Tensor out;
    {
        const NoGil no_gil;
        out = record ? run_recorded(c, keep != 0) : run_forward(c, nullptr);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// backward(q, k, v, mask, dout, T, B, pre_pad, variant, flags) -> (dq, dk, dv) or None
PyObject* py_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    Tensor dout;
    if (n != 10 || !tensor(args[0], &c.q) || !tensor(args[1], &c.k) || !tensor(args[2], &c.v) || !tensor_or_none(args[3], &c.mask) ||
        !tensor(args[4], &dout) || !scalars(args + 5, &c) || !valid(c) || dout.sizes() != c.v.sizes() || dout.device() != c.v.device())
        Py_RETURN_NONE;
    Grads g;
    {
        const NoGil no_gil;
        const c10::AutoGradMode no_grad(false);
        g = run_backward(c, dout, Tensor());
    }
    PyObject* r = PyTuple_New(3);
    if (!r) throw python_error();
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(g.dq)));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(g.dk)));
    PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(std::move(g.dv)));
    return r;
    END_HANDLE_TH_ERRORS
}

// matrix(q, k, mask, T, B, pre_pad, variant, flags) -> (E, H, N, N) fp32 Tensor or None
PyObject* py_matrix(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    if (n != 8 || !tensor(args[0], &c.q) || !tensor(args[1], &c.k) || !tensor_or_none(args[2], &c.mask) || !scalars(args + 3, &c))
        Py_RETURN_NONE;
    c.v = c.q;
    if (!valid(c)) Py_RETURN_NONE;
    Tensor A;
    {
        const NoGil no_gil;
        A = run_matrix(c);
    }
    return THPVariable_Wrap(std::move(A));
    END_HANDLE_TH_ERRORS
}

// workspaces() -> list of the cached workspace buffers
PyObject* py_workspaces(PyObject*, PyObject*) {
    HANDLE_TH_ERRORS
    std::vector<Tensor> buffers;
    {
        const NoGil no_gil;
        std::vector<std::shared_ptr<Workspace>> all;
        {
            const std::lock_guard<std::mutex> lock(g_mutex);
            for (const auto& kv : g_workspaces) all.push_back(kv.second);
        }
        for (const auto& w : all) {
            const std::lock_guard<std::mutex> lock(w->lock);
            if (w->buf.defined()) buffers.push_back(w->buf);
        }
    }
    PyObject* r = PyList_New(0);
    if (!r) throw python_error();
    for (const Tensor& buf : buffers) {
        PyObject* t = THPVariable_Wrap(buf);
        PyList_Append(r, t);
        Py_DECREF(t);
    }
    return r;
    END_HANDLE_TH_ERRORS
}

PyObject* py_clear(PyObject*, PyObject*) {
    HANDLE_TH_ERRORS
    {
        const NoGil no_gil;
        std::map<std::pair<int, void*>, std::shared_ptr<Workspace>> gone;
        const std::lock_guard<std::mutex> lock(g_mutex);
        gone.swap(g_workspaces);
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// bind(path): look the entry points up in the library
PyObject* py_bind(PyObject*, PyObject* arg) {
    const char* path = PyUnicode_AsUTF8(arg);
    if (!path) return nullptr;
    void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!lib) return PyErr_Format(PyExc_ImportError, "%s", dlerror());
    const struct { void** slot; const char* name; } want[] = {
        {reinterpret_cast<void**>(&api.strerror), "ma_strerror"},
        {reinterpret_cast<void**>(&api.layout), "ma_fwd_workspace_layout"},
        {reinterpret_cast<void**>(&api.workspace_bytes), "ma_fwd_workspace_bytes"},
        {reinterpret_cast<void**>(&api.fwd), "ma_fwd"},
        {reinterpret_cast<void**>(&api.state_bytes), "ma_fwd_state_bytes"},
        {reinterpret_cast<void**>(&api.keep_workspace_bytes), "ma_fwd_keep_workspace_bytes"},
        {reinterpret_cast<void**>(&api.fwd_keep), "ma_fwd_keep"},
        {reinterpret_cast<void**>(&api.matrix_workspace_bytes), "ma_matrix_workspace_bytes"},
        {reinterpret_cast<void**>(&api.matrix), "ma_matrix"},
        {reinterpret_cast<void**>(&api.bwd_workspace_bytes), "ma_bwd_workspace_bytes"},
        {reinterpret_cast<void**>(&api.bwd), "ma_bwd"},
        {reinterpret_cast<void**>(&api.bwd_kept_workspace_bytes), "ma_bwd_kept_workspace_bytes"},
        {reinterpret_cast<void**>(&api.bwd_kept), "ma_bwd_kept"},
    };
    for (const auto& w : want)
        if ((*w.slot = dlsym(lib, w.name)) == nullptr) return PyErr_Format(PyExc_ImportError, "%s does not export %s", path, w.name);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_O, nullptr},
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_forward)), METH_FASTCALL, nullptr},
    {"backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_backward)), METH_FASTCALL, nullptr},
    {"matrix", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_matrix)), METH_FASTCALL, nullptr},
    {"workspaces", py_workspaces, METH_NOARGS, nullptr},
    {"clear", py_clear, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ma_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ma_host(void) { return PyModule_Create(&module); }
