// Host path of the operators behind torch: from the Python call to the C ABI without Python in between.
//
// A call on a short sequence is bound by its host side: the GPU needs 18 us for a forward of one head of 640 positions and
// 50-160 us for a training step of a small model, while the Python wrappers (tensor checks, a torch.empty per output, ctypes
// with 20 arguments, autograd.Function in the engine's thread) took 36 and 230 us.  Here the checks read the tensors' fields,
// the allocations go to torch's caching allocator directly, what a training step keeps for its backward shares one of them, and
// the backward is a C++ node, which the autograd engine's thread runs without the interpreter lock.
//
// Every function takes the operator's tensors and returns its result, or None for whatever the fast path does not serve
// (unusual layouts, padded or widened head dimensions, arguments that are an error, calls under a function transform, a tracer,
// a dispatch mode or with forward-mode tangents): the Python wrappers then do what they always did, error messages included.
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/version.h>
#include <algorithm>
#include <vector>
#include "mlstm_train.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// Raises what the Python wrappers raise for a return code of the library.
[[noreturn]] void raise_python(PyObject* type, const std::string& text) {
    PyGILState_STATE gil = PyGILState_Ensure();
    PyErr_SetString(type, text.c_str());
    python_error err;
    err.persist();
    PyGILState_Release(gil);
    throw std::move(err);
}
void check_rc(int rc, const char* what) {
    if (rc == 0) return;
    if (rc > 0) raise_python(PyExc_RuntimeError, std::string(what) + ": HIP error " + std::to_string(rc));
    const char* text = "error";
    switch (rc) {
        case MLSTM_EINVAL: text = "invalid argument (null pointer, non-positive size or unknown dtype)"; break;
        case MLSTM_ESHAPE: text = "unsupported shape (head dimension / sequence length)"; break;
        case MLSTM_EWORKSPACE: text = "workspace (or saved buffer) too small or of the wrong size"; break;
        case MLSTM_EKERNEL: text = "a kernel's bounded wait expired"; break;
        case MLSTM_ESAVED: text = "a backward was given a saved buffer written for another shape or setting"; break;
        case MLSTM_EBUILD: text = "a kernel with hand-counted memory waits was compiled with register spills"; break;
    }
    raise_python(PyExc_ValueError, std::string(what) + ": " + text + " (code " + std::to_string(rc) + ")");
}

void* hip_stream() { return c10::hip::getCurrentHIPStream().stream(); }

int type_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return MLSTM_F32;
        case at::kHalf: return MLSTM_F16;
        case at::kBFloat16: return MLSTM_BF16;
        default: return -1;
    }
}

// Device memory of the call's stream, given back to the caching allocator when it goes out of scope.
struct Buffer {
    at::DataPtr p;
    size_t n = 0;
    explicit Buffer(size_t bytes) : n(bytes) {
        if (bytes) p = c10::GetAllocator(c10::kCUDA)->allocate(bytes);
    }
    Buffer() = default;
    void* get(size_t off = 0) const { return n ? static_cast<char*>(p.get()) + off : nullptr; }
};
Tensor new_tensor(at::IntArrayRef size, at::IntArrayRef stride, at::ScalarType type, const Tensor& like) {
    return Tensor(at::detail::empty_strided_cuda(size, stride, type, like.device()));
}
Tensor new_like(const Tensor& t) { return new_tensor(t.sizes(), t.strides(), t.scalar_type(), t); }
// A new tensor of t's shape ([B,NH,S,D], D contiguous), dense in the order of t's dimensions in memory.
Tensor dense_in_order_of(const Tensor& t) {
    int order[3] = {0, 1, 2};
    auto key = [&](int d) { return std::pair<int64_t, int>(t.stride(d), t.size(d) == 1 ? -d : 0); };
    std::stable_sort(order, order + 3, [&](int a, int b) { return key(a) > key(b); });
    int64_t strides[4], step = t.size(3);
    strides[3] = 1;
    for (int n = 2; n >= 0; n--) { strides[order[n]] = step; step *= t.size(order[n]); }
    return new_tensor(t.sizes(), at::IntArrayRef(strides, 4), t.scalar_type(), t);
}
// dh in h's layout (the kernels read h and dh through one set of strides)
Tensor like_layout(const Tensor& t, const Tensor& h) {
    if (t.strides() == h.strides()) return t;
    Tensor out = new_tensor(h.sizes(), h.strides(), t.scalar_type(), t);
    out.copy_(t);
    return out;
}
// Does the view address one element more than once?  (The test of the library for tensors it writes.)
bool overlaps(const Tensor& t) {
    int n = 0;
    std::pair<int64_t, int64_t> d[8];
    for (int64_t k = 0; k < t.dim() && n < 8; k++)
        if (t.size(k) > 1) d[n++] = {t.stride(k), t.size(k)};
    std::sort(d, d + n);
    int64_t extent = 1;
    for (int k = 0; k < n; k++) {
        if (d[k].first < extent) return true;
        extent += (d[k].second - 1) * d[k].first;
    }
    return false;
}

struct Call {
    int B = 0, NH = 0, S = 0, D = 0, dtype = 0, gate_dtype = 0, gate_form = 0;
    mlstm_layout layout(const Tensor& q, const Tensor& h, const Tensor& f) const {
        return mlstm_layout{q.stride(0), q.stride(1), q.stride(2), h.stride(0), h.stride(1), h.stride(2), f.stride(0), f.stride(1), f.stride(2), gate_form};
    }
    bool on_tiles() const { return D == 64 || D == 128; }   // scan form: the head dimensions that the tile kernels serve
    bool operator==(const Call& x) const {
        return B == x.B && NH == x.NH && S == x.S && D == x.D && dtype == x.dtype && gate_dtype == x.gate_dtype && gate_form == x.gate_form;
    }
    size_t kept_bytes() const { return mlstm::train_kept_bytes(B, NH, S, D, dtype); }
    Buffer workspace(int op) const { return Buffer(mlstm_workspace_bytes(op, B, NH, S, D, dtype)); }
};

// Is this a call of the matmul form that goes to the library as it is?  q, k, v of one shape, type and layout, gates of one
// type and layout, everything on the current device, no view that addresses an element twice.
bool takes_matmul(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& f, const Tensor& i, int precise, int gate_form, Call& c) {
    if (q.dim() != 4 || f.dim() != 3) return false;
    if (k.sizes() != q.sizes() || v.sizes() != q.sizes() || i.sizes() != f.sizes()) return false;
    if (k.strides() != q.strides() || v.strides() != q.strides() || i.strides() != f.strides()) return false;
    const auto type = q.scalar_type();
    if (k.scalar_type() != type || v.scalar_type() != type || i.scalar_type() != f.scalar_type()) return false;
    c.B = (int)q.size(0); c.NH = (int)q.size(1); c.S = (int)q.size(2); c.D = (int)q.size(3);
    if (f.size(0) != c.B || f.size(1) != c.NH || f.size(2) != c.S || q.numel() == 0 || q.size(2) > (1 << 20) || q.size(0) * q.size(1) > (1 << 30)) return false;
    const int t = type_code(type), g = type_code(f.scalar_type());
    if (t < 0 || g < 0) return false;
    if (!(c.D == 64 || c.D == 128 || c.D == 256 || (t == MLSTM_F32 && (c.D == 512 || c.D == 1024)))) return false;
    if (q.stride(3) != 1 || overlaps(q) || overlaps(f)) return false;
    c.dtype = t | (precise && t != MLSTM_F32 ? MLSTM_PRECISE : 0);
    c.gate_dtype = g;
    c.gate_form = gate_form;
    return true;
}

// The nodes of the graph: the inputs, what else the backward reads (`own`: a buffer of the library's, the ungated output) and
// an output it reads, all as saved variables: under autograd's version checks and its saved-tensor hooks (checkpointing,
// offloading), which may hand back other tensors of the same values.
struct OpNode : torch::autograd::Node {
    Call c;
    std::vector<SavedVariable> vars, own;
    SavedVariable out;
    void save(std::initializer_list<Tensor> ts) {
        vars.reserve(ts.size());
        for (const Tensor& t : ts) vars.emplace_back(t, false);
    }
    void save_own(std::initializer_list<Tensor> ts) {
        own.reserve(ts.size());
        for (const Tensor& t : ts) own.emplace_back(t, false);
    }
    void release_variables() override {
        for (auto& v : vars) v.reset_data();
        for (auto& v : own) v.reset_data();
        out.reset_data();
    }
    static std::vector<Tensor> unpack(std::vector<SavedVariable>& from) {
        std::vector<Tensor> ts;
        ts.reserve(from.size());
        for (auto& v : from) ts.push_back(v.unpack());
        return ts;
    }
    std::vector<Tensor> inputs() { return unpack(vars); }
};
[[noreturn]] void saved_changed() { raise_python(PyExc_RuntimeError, "a tensor saved for the backward came back with another shape, type or device"); }
// a tensor of these sizes and type, dense, on a 16-byte boundary, with the values of a saved one
Tensor dense_saved(const Tensor& t, at::IntArrayRef sizes, at::ScalarType type, const at::Device& device) {
    if (t.device() != device || t.scalar_type() != type || t.sizes() != sizes) saved_changed();
    Tensor d = t.contiguous();
    return reinterpret_cast<size_t>(d.data_ptr()) & 15 ? d.clone() : d;
}
Tensor bytes_tensor(size_t n, const Tensor& like) { return new_tensor({(int64_t)n}, {1}, at::kByte, like); }
Tensor kept_saved(const Tensor& t, const Tensor& like) { return dense_saved(t, {t.dim() == 1 ? t.size(0) : -1}, at::kByte, like.device()); }
template <typename N, typename... T>
std::shared_ptr<N> make_node(const T&... inputs) {
    std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(inputs...));
    return node;
}
template <typename... T>
bool wants_grad(const T&... ts) { return at::GradMode::is_enabled() && (ts.requires_grad() || ...); }

void contiguous_head(const Tensor& dh) {
    if (dh.stride(-1) != 1 && dh.size(-1) != 1) raise_python(PyExc_AssertionError, "dh must have a contiguous head dimension");
}
// the checks of an output gradient that the autograd engine has not made already
void same_type(const Tensor& dh, const Tensor& q) {
    if (dh.scalar_type() != q.scalar_type()) raise_python(PyExc_TypeError, "dh must have q's dtype");
}

// the saved q, k, v, f, i of the matmul form: as they were, or dense copies where a hook changed their layouts
void matmul_inputs(std::vector<Tensor>& in, const Call& c) {
    for (const Tensor& t : in)
        if (t.device() != in[0].device() || !t.is_cuda()) saved_changed();
    Call now;
    const int precise = c.dtype & MLSTM_PRECISE ? 1 : 0;
    if (!takes_matmul(in[0], in[1], in[2], in[3], in[4], precise, c.gate_form, now)) {
        for (int n = 0; n < 5; n++) in[n] = in[n].contiguous();
        if (!takes_matmul(in[0], in[1], in[2], in[3], in[4], precise, c.gate_form, now)) saved_changed();
    }
    if (!(now == c)) saved_changed();
}
// the saved output (or ungated output), in its layout where that is one the kernels address
Tensor rows_saved(const Tensor& h, const Tensor& q) {
    if (h.device() != q.device() || h.scalar_type() != q.scalar_type() || h.sizes() != q.sizes()) saved_changed();
    return h.stride(3) != 1 || overlaps(h) ? h.contiguous() : h;
}

// ---- matmul form ------------------------------------------------------------------------------------------------------

struct Triton_mLSTMBackward : OpNode {
    std::string name() const override { return "Triton_mLSTMBackward"; }
    variable_list apply(variable_list&& grads) override {
        variable_list res(5);
        at::NoGradGuard no_grad;
        auto in = inputs();
        matmul_inputs(in, c);
        const Tensor h = rows_saved(out.unpack(getptr()), in[0]), kept = kept_saved(own[0].unpack(), h);
        Tensor dh = grads[0].defined() ? grads[0] : at::zeros_like(h);
        contiguous_head(dh);
        same_type(dh, in[0]);
        dh = like_layout(dh, h);
        for (int n = 0; n < 5; n++) res[n] = new_like(in[n]);
        const mlstm_layout lay = c.layout(in[0], h, in[3]);
        Buffer ws = c.workspace(MLSTM_OP_BACKWARD);
        check_rc(mlstm::train_backward(dh.data_ptr(), in[0].data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(), nullptr,
                                       h.data_ptr(), kept.data_ptr(), kept.numel(), res[0].data_ptr(), res[1].data_ptr(), res[2].data_ptr(), res[3].data_ptr(),
                                       res[4].data_ptr(), nullptr, c.B, c.NH, c.S, c.D, c.dtype, c.gate_dtype, &lay, ws.get(), ws.n, hip_stream()),
                 "mlstm_backward_saved_lx");
        return res;
    }
};

bool matmul(const Tensor* t, int precise, int gate_form, bool train, Tensor& h) {
    const Tensor &q = t[0], &k = t[1], &v = t[2], &f = t[3], &i = t[4];
    Call c;
    if (!takes_matmul(q, k, v, f, i, precise, gate_form, c)) return false;
    h = dense_in_order_of(q);
    const mlstm_layout lay = c.layout(q, h, f);
    Buffer ws = c.workspace(MLSTM_OP_FORWARD);
    if (!train || !wants_grad(q, k, v, f, i)) {
        check_rc(mlstm_forward_lx(q.data_ptr(), k.data_ptr(), v.data_ptr(), f.data_ptr(), i.data_ptr(), h.data_ptr(), nullptr, nullptr, c.B, c.NH, c.S, c.D,
                                  c.dtype, c.gate_dtype, &lay, ws.get(), ws.n, hip_stream()),
                 "mlstm_forward_lx");
        return true;
    }
    auto node = make_node<Triton_mLSTMBackward>(q, k, v, f, i);
    node->c = c;
    const Tensor kept = bytes_tensor(c.kept_bytes(), q);
    check_rc(mlstm::train_forward(q.data_ptr(), k.data_ptr(), v.data_ptr(), f.data_ptr(), i.data_ptr(), nullptr, h.data_ptr(), nullptr, kept.data_ptr(),
                                  kept.numel(), c.B, c.NH, c.S, c.D, c.dtype, c.gate_dtype, &lay, ws.get(), ws.n, hip_stream()),
             "mlstm_forward_save_lx");
    node->save({q, k, v, f, i});
    node->save_own({kept});
    torch::autograd::set_history(h, node);
    node->out = SavedVariable(h, true);
    return true;
}

// ---- matmul form with the output gate ---------------------------------------------------------------------------------

struct Triton_mLSTM_gatedBackward : OpNode {
    std::string name() const override { return "Triton_mLSTM_gatedBackward"; }
    variable_list apply(variable_list&& grads) override {
        variable_list res(6);
        at::NoGradGuard no_grad;
        auto in = inputs();
        matmul_inputs(in, c);
        const Tensor h = rows_saved(own[1].unpack(), in[0]), kept = kept_saved(own[0].unpack(), h);
        if (in[5].device() != h.device() || in[5].scalar_type() != h.scalar_type() || in[5].sizes() != h.sizes()) saved_changed();
        Tensor dh = grads[0].defined() ? grads[0] : at::zeros_like(h);
        contiguous_head(dh);
        same_type(dh, in[0]);
        dh = like_layout(dh, h);
        const Tensor o = like_layout(in[5], h);
        for (int n = 0; n < 5; n++) res[n] = new_like(in[n]);
        res[5] = new_like(h);
        const mlstm_layout lay = c.layout(in[0], h, in[3]);
        Buffer ws = c.workspace(MLSTM_OP_BACKWARD_GATED);
        check_rc(mlstm::train_backward(dh.data_ptr(), in[0].data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                       o.data_ptr(), h.data_ptr(), kept.data_ptr(), kept.numel(), res[0].data_ptr(), res[1].data_ptr(), res[2].data_ptr(), res[3].data_ptr(),
                                       res[4].data_ptr(), res[5].data_ptr(), c.B, c.NH, c.S, c.D, c.dtype, c.gate_dtype, &lay, ws.get(), ws.n,
                                       hip_stream()),
                 "mlstm_backward_gated_lx");
        return res;
    }
};

bool gated(const Tensor* t, bool train, Tensor& hg) {
    const Tensor &q = t[0], &k = t[1], &v = t[2], &f = t[3], &i = t[4];
    Call c;
    if (!takes_matmul(q, k, v, f, i, 0, MLSTM_GATE_RAW, c)) return false;
    if (t[5].sizes() != q.sizes() || t[5].scalar_type() != q.scalar_type()) return false;
    Tensor h = dense_in_order_of(q);
    hg = new_like(h);
    const bool keep = train && wants_grad(q, k, v, f, i, t[5]);
    Tensor o;
    {
        at::NoGradGuard no_grad;
        o = like_layout(t[5], h);
    }
    const mlstm_layout lay = c.layout(q, h, f);
    Buffer ws = c.workspace(MLSTM_OP_FORWARD_GATED);
    if (!keep) {
        check_rc(mlstm_forward_gated_lx(q.data_ptr(), k.data_ptr(), v.data_ptr(), f.data_ptr(), i.data_ptr(), o.data_ptr(), h.data_ptr(), hg.data_ptr(),
                                        nullptr, nullptr, c.B, c.NH, c.S, c.D, c.dtype, c.gate_dtype, &lay, ws.get(), ws.n, hip_stream()),
                 "mlstm_forward_gated_lx");
        return true;
    }
    auto node = make_node<Triton_mLSTM_gatedBackward>(q, k, v, f, i, t[5]);
    node->c = c;
    const Tensor kept = bytes_tensor(c.kept_bytes(), q);
    check_rc(mlstm::train_forward(q.data_ptr(), k.data_ptr(), v.data_ptr(), f.data_ptr(), i.data_ptr(), o.data_ptr(), h.data_ptr(), hg.data_ptr(),
                                  kept.data_ptr(), kept.numel(), c.B, c.NH, c.S, c.D, c.dtype, c.gate_dtype, &lay, ws.get(), ws.n, hip_stream()),
             "mlstm_forward_gated_lx");
    node->save({q, k, v, f, i, t[5]});
    node->save_own({kept, h});
    torch::autograd::set_history(hg, node);
    return true;
}

// ---- scan form --------------------------------------------------------------------------------------------------------

struct Scan_mLSTMBackward : OpNode {
    std::string name() const override { return "Scan_mLSTMBackward"; }
    variable_list apply(variable_list&& grads) override {
        variable_list res(6);
        at::NoGradGuard no_grad;
        auto in = inputs();
        const at::Device device = in[0].device();
        if (!device.is_cuda()) saved_changed();
        const int64_t rows[4] = {c.B, c.NH, c.S, c.D};
        for (int n = 0; n < 6; n++) {
            in[n] = dense_saved(in[n], at::IntArrayRef(rows, n == 3 || n == 4 ? 3 : 4), at::kFloat, device);
            res[n] = new_like(in[n]);
        }
        const Tensor kept = kept_saved(own[0].unpack(), in[0]), h_ungated = dense_saved(own[1].unpack(), at::IntArrayRef(rows, 4), at::kFloat, device);
        if (grads[0].defined() && grads[0].scalar_type() != at::kFloat) raise_python(PyExc_TypeError, "dh must be float32");
        const Tensor dh = grads[0].defined() ? dense_saved(grads[0], at::IntArrayRef(rows, 4), at::kFloat, device) : at::zeros_like(in[0]);
        if (c.on_tiles()) {
            Buffer ws = c.workspace(MLSTM_OP_BACKWARD_GATED);
            check_rc(mlstm::train_backward(dh.data_ptr(), in[0].data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                           in[5].data_ptr(), h_ungated.data_ptr(), kept.data_ptr(), kept.numel(), res[0].data_ptr(), res[1].data_ptr(), res[2].data_ptr(),
                                           res[3].data_ptr(), res[4].data_ptr(), res[5].data_ptr(), c.B, c.NH, c.S, c.D, MLSTM_F32, MLSTM_F32, nullptr,
                                           ws.get(), ws.n, hip_stream()),
                     "mlstm_scan_backward_saved_ex");
            return res;
        }
        if (kept.numel() != 4ll * c.B * c.NH * c.S) saved_changed();
        Buffer ws = c.workspace(MLSTM_OP_SCAN_BACKWARD);
        check_rc(mlstm_scan_backward_saved_ex(dh.data_ptr(), in[0].data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                              in[5].data_ptr(), h_ungated.data_ptr(), static_cast<float*>(kept.data_ptr()), res[0].data_ptr(), res[1].data_ptr(), res[2].data_ptr(),
                                              res[3].data_ptr(), res[4].data_ptr(), res[5].data_ptr(), c.B, c.NH, c.S, c.D, MLSTM_F32, ws.get(), ws.n,
                                              hip_stream()),
                 "mlstm_scan_backward_saved_ex");
        return res;
    }
};

bool scan(const Tensor* t, Tensor& h) {
    const Tensor& q = t[0];
    if (q.dim() != 4 || q.numel() == 0) return false;
    Call c;
    c.B = (int)q.size(0); c.NH = (int)q.size(1); c.S = (int)q.size(2); c.D = (int)q.size(3);
    Tensor in[6];
    const bool keep = wants_grad(t[0], t[1], t[2], t[3], t[4], t[5]);
    {
        at::NoGradGuard no_grad;
        for (int n = 0; n < 6; n++) {
            const bool gate = n == 3 || n == 4;
            if (t[n].scalar_type() != at::kFloat || (gate ? t[n].sizes() != q.sizes().slice(0, 3) : t[n].sizes() != q.sizes())) return false;
            in[n] = t[n].contiguous();   // (on a 16-byte boundary: the kernels copy whole rows of 16-byte pieces into LDS)
            if (reinterpret_cast<size_t>(in[n].data_ptr()) & 15) in[n] = in[n].clone();
        }
    }
    h = new_like(in[0]);
    if (!keep) {
        Buffer ws = c.workspace(MLSTM_OP_SCAN_FORWARD);
        check_rc(mlstm_scan_forward_ex(in[0].data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(), in[5].data_ptr(),
                                       h.data_ptr(), c.B, c.NH, c.S, c.D, MLSTM_F32, ws.get(), ws.n, hip_stream()),
                 "mlstm_scan_forward_ex");
        return true;
    }
    auto node = make_node<Scan_mLSTMBackward>(t[0], t[1], t[2], t[3], t[4], t[5]);
    node->c = c;
    const Tensor h_ungated = new_like(in[0]);
    Tensor kept;
    if (c.on_tiles()) {
        kept = bytes_tensor(c.kept_bytes(), h);
        Buffer ws = c.workspace(MLSTM_OP_FORWARD_GATED);
        check_rc(mlstm::train_forward(in[0].data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(), in[5].data_ptr(),
                                      h_ungated.data_ptr(), h.data_ptr(), kept.data_ptr(), kept.numel(), c.B, c.NH, c.S, c.D, MLSTM_F32, MLSTM_F32, nullptr,
                                      ws.get(), ws.n, hip_stream()),
                 "mlstm_scan_forward_save_ex");
    } else {
        kept = bytes_tensor((size_t)c.B * c.NH * c.S * 4, h);   // the normaliser sums
        Buffer ws = c.workspace(MLSTM_OP_SCAN_FORWARD);
        check_rc(mlstm_scan_forward_save_ex(in[0].data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(), in[5].data_ptr(),
                                            h.data_ptr(), h_ungated.data_ptr(), static_cast<float*>(kept.data_ptr()), c.B, c.NH, c.S, c.D,
                                            MLSTM_F32, ws.get(), ws.n, hip_stream()),
                 "mlstm_scan_forward_save_ex");
    }
    node->save({t[0], t[1], t[2], t[3], t[4], t[5]});
    node->save_own({kept, h_ungated});
    torch::autograd::set_history(h, node);
    return true;
}

// ---- sLSTM ------------------------------------------------------------------------------------------------------------

struct HIP_sLSTMBackward : OpNode {
    int forget_sigmoid = 0;
    std::string name() const override { return "HIP_sLSTMBackward"; }
    variable_list apply(variable_list&& grads) override {
        variable_list res(3);
        at::NoGradGuard no_grad;
        auto in = inputs();   // r alone: the pre-activations of wx are in the saved states
        const Tensor h_saved = out.unpack(getptr());
        const at::Device device = h_saved.device();
        if (!device.is_cuda()) saved_changed();
        const int64_t rows[4] = {c.B, c.S, c.NH, c.D}, mats[4] = {c.NH, 4, c.D, c.D};
        const Tensor h = dense_saved(h_saved, at::IntArrayRef(rows, 4), at::kFloat, device), r = dense_saved(in[0], at::IntArrayRef(mats, 4), at::kFloat, device);
        const Tensor kept = kept_saved(own[0].unpack(), h);
        if ((size_t)kept.numel() != slstm_saved_bytes(c.B, c.NH, c.S, c.D)) saved_changed();
        if (grads[0].defined() && grads[0].scalar_type() != at::kFloat) raise_python(PyExc_TypeError, "dh must be float32");
        const Tensor dh = grads[0].defined() ? grads[0].contiguous() : at::zeros_like(h);
        const int64_t wx[5] = {c.B, c.S, 4, c.NH, c.D}, sx[5] = {4ll * c.S * c.NH * c.D, 4ll * c.NH * c.D, (int64_t)c.NH * c.D, c.D, 1};
        const int64_t bs[3] = {c.NH, 4, c.D}, sb[3] = {4ll * c.D, c.D, 1};
        res[0] = new_tensor(at::IntArrayRef(wx, 5), at::IntArrayRef(sx, 5), at::kFloat, h);
        res[1] = new_like(r);
        res[2] = new_tensor(at::IntArrayRef(bs, 3), at::IntArrayRef(sb, 3), at::kFloat, h);
        Buffer ws(slstm_workspace_bytes(c.B, c.NH, c.S, c.D));
        check_rc(slstm_backward_ex(dh.data_ptr<float>(), h.data_ptr<float>(), r.data_ptr<float>(), static_cast<const float*>(kept.data_ptr()),
                                   res[0].data_ptr<float>(), res[1].data_ptr<float>(), res[2].data_ptr<float>(), c.B, c.NH, c.S, c.D, forget_sigmoid,
                                   ws.get(), ws.n, hip_stream()),
                 "slstm_backward_ex");
        return res;
    }
};

bool slstm(const Tensor* t, int forget_sigmoid, Tensor& h) {
    const Tensor &wx = t[0], &r = t[1], &b = t[2];
    if (wx.dim() != 5 || wx.size(2) != 4 || wx.numel() == 0 || r.dim() != 4 || b.dim() != 3) return false;
    Call c;
    c.B = (int)wx.size(0); c.S = (int)wx.size(1); c.NH = (int)wx.size(3); c.D = (int)wx.size(4);
    if (!(c.D == 32 || c.D == 64 || c.D == 128)) return false;
    if (r.size(0) != c.NH || r.size(1) != 4 || r.size(2) != c.D || r.size(3) != c.D || b.size(0) != c.NH || b.size(1) != 4 || b.size(2) != c.D) return false;
    for (int n = 0; n < 3; n++)
        if (t[n].scalar_type() != at::kFloat || !t[n].is_contiguous()) return false;
    const int64_t hs[4] = {c.B, c.S, c.NH, c.D}, sh[4] = {(int64_t)c.S * c.NH * c.D, (int64_t)c.NH * c.D, c.D, 1};
    h = new_tensor(at::IntArrayRef(hs, 4), at::IntArrayRef(sh, 4), at::kFloat, wx);
    const bool keep = wants_grad(wx, r, b);
    std::shared_ptr<HIP_sLSTMBackward> node;
    Tensor kept;
    if (keep) {
        node = make_node<HIP_sLSTMBackward>(wx, r, b);
        node->c = c;
        node->forget_sigmoid = forget_sigmoid;
        kept = bytes_tensor(slstm_saved_bytes(c.B, c.NH, c.S, c.D), wx);
    }
    check_rc(slstm_forward_ex(wx.data_ptr<float>(), r.data_ptr<float>(), b.data_ptr<float>(), h.data_ptr<float>(),
                              keep ? static_cast<float*>(kept.data_ptr()) : nullptr, c.B, c.NH, c.S, c.D, forget_sigmoid, hip_stream()),
             "slstm_forward_ex");
    if (keep) {
        node->save({r});
        node->save_own({kept});
        torch::autograd::set_history(h, node);
        node->out = SavedVariable(h, true);
    }
    return true;
}

// ---- Python -----------------------------------------------------------------------------------------------------------

// The first `n` arguments as plain tensors on the current device (false: something else is among them).
// Calls that a dispatch mode, a tracer or a function transform would have to see are not served here, nor forward-mode tangents.
bool tensors(PyObject* const* args, Py_ssize_t nargs, int n, Tensor* t) {
    if (nargs < n || c10::impl::dispatch_mode_enabled() || at::tracer::impl::is_dispatch_enabled() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return false;
    for (int k = 0; k < n; k++) {
        if (!THPVariable_CheckExact(args[k])) return false;
        t[k] = THPVariable_Unpack(args[k]);
        if (!t[k].is_cuda() || t[k].layout() != at::kStrided) return false;
        if (t[k]._fw_grad(0).defined()) return false;
    }
    const auto dev = t[0].device();
    if (dev.index() != c10::hip::current_device()) return false;
    for (int k = 1; k < n; k++)
        if (t[k].device() != dev) return false;
    return true;
}
int flag(PyObject* const* args, Py_ssize_t nargs, int k) { return nargs > k ? (int)PyLong_AsLong(args[k]) : 0; }
PyObject* result(bool served, const Tensor& t) {
    if (!served) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}

// (q, k, v, f, i, precise, gate_form): h, no graph
PyObject* py_matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Tensor t[5], h;
    return result(tensors(args, nargs, 5, t) && matmul(t, flag(args, nargs, 5), flag(args, nargs, 6), false, h), h);
    END_HANDLE_TH_ERRORS
}
// (q, k, v, f, i, precise, gate_form): h, with a graph where one is wanted
PyObject* py_matmul_train(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Tensor t[5], h;
    return result(tensors(args, nargs, 5, t) && matmul(t, flag(args, nargs, 5), flag(args, nargs, 6), true, h), h);
    END_HANDLE_TH_ERRORS
}
// (q, k, v, f, i, o): silu(o) * h, no graph
PyObject* py_gated(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Tensor t[6], h;
    return result(tensors(args, nargs, 6, t) && gated(t, false, h), h);
    END_HANDLE_TH_ERRORS
}
PyObject* py_gated_train(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Tensor t[6], h;
    return result(tensors(args, nargs, 6, t) && gated(t, true, h), h);
    END_HANDLE_TH_ERRORS
}
// (q, k, v, f, i, o): the scan form, with a graph where one is wanted
PyObject* py_scan(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Tensor t[6], h;
    return result(tensors(args, nargs, 6, t) && scan(t, h), h);
    END_HANDLE_TH_ERRORS
}
// (wx, r, b, forget_sigmoid): the sLSTM cell, with a graph where one is wanted
PyObject* py_slstm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Tensor t[3], h;
    return result(tensors(args, nargs, 3, t) && slstm(t, flag(args, nargs, 3), h), h);
    END_HANDLE_TH_ERRORS
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL, nullptr
PyMethodDef methods[] = {{"matmul", FAST(py_matmul)},           {"matmul_train", FAST(py_matmul_train)}, {"gated", FAST(py_gated)},
                         {"gated_train", FAST(py_gated_train)}, {"scan", FAST(py_scan)},                 {"slstm", FAST(py_slstm)},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// (torch_version: the release whose headers this was built with; a tensor's layout in memory belongs to one of them)
PyMODINIT_FUNC PyInit__native(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
