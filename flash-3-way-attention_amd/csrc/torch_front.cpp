// The path from a torch tensor to the C ABI in native code: what the Python autograd Functions of this package do per call
// (checks, layouts, outputs, workspace, the library call, and the same again in the backward) as C++ autograd Functions.
//
// Why: a call at the small configurations is a few launches of 5-50 us on the GPU, and the Python host path took longer than
// they do (a ctypes call with thirty arguments, five to ten allocations and a dozen tensor queries from the interpreter; for
// the backward also the hand-over of the engine's thread to the interpreter): 38 us per forward, 100-130 us per backward.
//
// tdp() and dps() take the usual case only and return None for everything else -- tensors that are not plain GPU tensors
// (subclasses, wrappers, tangents), shapes, types or windows that do not fit, calls under a functorch transform or a
// tracer -- which the Python Functions then handle or refuse as they always did.  Nothing is computed here and nothing is
// kept between calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include <array>
#include <optional>
#include <stdexcept>
#include <string>

#include "../../include/trittention_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

int dtype_code(at::ScalarType t) {
    return t == at::kFloat ? TRITT_F32 : t == at::kBFloat16 ? TRITT_BF16 : t == at::kHalf ? TRITT_F16 : -1;
}

// Whether the library can read `t` where it lies (tritt_layout's contract): dense last dimension, every other stride a
// non-negative multiple of 16 bytes, 16-byte aligned start.
bool viewable(const Tensor& t) {
    const int64_t unit = 16 / (int64_t)t.element_size();
    if ((t.size(3) > 1 && t.stride(3) != 1) || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) return false;
    for (int i = 0; i < 3; ++i)
        if (t.size(i) != 1 && (t.stride(i) < 0 || t.stride(i) % unit)) return false;
    return true;
}
Tensor view(const Tensor& t) {
    if (viewable(t)) return t;
    Tensor d = t.contiguous();
    return reinterpret_cast<uintptr_t>(d.data_ptr()) % 16 ? d.clone(at::MemoryFormat::Contiguous) : d;
}
tritt_layout layout_of(const Tensor& t) {
    auto s = [&](int i) { return t.size(i) > 1 ? (long long)t.stride(i) : 0LL; };
    return tritt_layout{s(0), s(1), s(2)};
}
struct Layouts {
    bool dense;
    std::array<tritt_layout, 5> at;
};
Layouts layouts_of(const std::array<Tensor, 5>& in) {
    Layouts l{true, {}};
    for (const Tensor& t : in) l.dense = l.dense && t.is_contiguous();
    if (!l.dense)
        for (int i = 0; i < 5; ++i) l.at[i] = layout_of(in[i]);
    return l;
}

void check(int status, const char* what) {
    if (status == TRITT_OK) return;
    throw std::runtime_error(std::string(what) + " failed: " + tritt_status_string(status) + " (status " +
                             std::to_string(status) + ")");
}
void* current_stream(const Tensor& t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream();
}
Tensor workspace(size_t bytes, const Tensor& like) {
    return at::empty({(int64_t)std::max<size_t>(bytes, 256)}, like.options().dtype(at::kByte));
}

struct Problem {
    double scale;
    bool causal;
    int64_t w[4];  // k1_window, k2_window, kk_left, kk_right; dot-product sum: k_diff in w[0]
    int64_t flags;
    bool keep = false;  // dot-product sum: the forward leaves what its backward would form again
};
void save(AutogradContext* ctx, const Problem& p) {
    ctx->saved_data["p"] = std::vector<int64_t>{p.causal, p.w[0], p.w[1], p.w[2], p.w[3], p.flags};
    ctx->saved_data["s"] = p.scale;
}
Problem load(AutogradContext* ctx) {
    const std::vector<int64_t> v = ctx->saved_data["p"].toIntVector();
    return Problem{ctx->saved_data["s"].toDouble(), v[0] != 0, {v[1], v[2], v[3], v[4]}, v[5]};
}
// a saved tensor as the library takes one that has to be dense (a saved-tensor hook may bring it back in another layout)
Tensor dense(const Tensor& t) {
    Tensor d = t.contiguous();
    return reinterpret_cast<uintptr_t>(d.data_ptr()) % 16 ? d.clone(at::MemoryFormat::Contiguous) : d;
}
Tensor gradient_like(const Tensor& q) { return at::empty(q.sizes(), q.options()); }

struct Tdp : torch::autograd::Function<Tdp> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k1_, const Tensor& k2_, const Tensor& v1_,
                          const Tensor& v2_, const Problem& p) {
        const std::array<Tensor, 5> in{view(q_), view(k1_), view(k2_), view(v1_), view(v2_)};
        const Tensor& q = in[0];
        const c10::OptionalDeviceGuard guard(q.device());
        const int B = (int)q.size(0), H = (int)q.size(1), T = (int)q.size(2), D = (int)q.size(3);
        const int code = dtype_code(q.scalar_type());
        const bool split = p.flags & TRITT_FLAG_SPLIT_OPERANDS;
        Tensor o = split ? at::empty({2, B, H, T, D}, q.options()) : gradient_like(q);
        Tensor lse = at::empty({B, H, T}, q.options().dtype(at::kFloat));
        const Layouts l = layouts_of(in);
        const int w1 = (int)p.w[0], w2 = (int)p.w[1], kl = (int)p.w[2], kr = (int)p.w[3];
        const unsigned flags = (unsigned)p.flags;
        const size_t need = l.dense ? tritt_tdp_fwd_workspace_bytes(B, H, T, D, code, p.causal, w1, w2, kl, kr, flags)
                                    : tritt_tdp_fwd_strided_workspace_bytes(B, H, T, D, code, p.causal, w1, w2, kl, kr, flags,
                                                                            l.at.data());
        const Tensor ws = workspace(need, q);
        void* st = current_stream(q);
        check(l.dense ? tritt_tdp_fwd(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                      o.data_ptr(), lse.data_ptr<float>(), B, H, T, D, code, (float)p.scale, p.causal, w1, w2,
                                      kl, kr, ws.data_ptr(), ws.numel(), flags, st)
                      : tritt_tdp_fwd_strided(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(),
                                              in[4].data_ptr(), l.at.data(), o.data_ptr(), lse.data_ptr<float>(), B, H, T, D,
                                              code, (float)p.scale, p.causal, w1, w2, kl, kr, ws.data_ptr(), ws.numel(), flags,
                                              st),
              "tritt_tdp_fwd");
        Tensor out = split ? o.select(0, 0) : o;  // split operands: the output and its rounding residual, both kept
        if (ctx) {
            ctx->save_for_backward({in[0], in[1], in[2], in[3], in[4], split ? o : out, lse});
            save(ctx, p);
        }
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grad) {
        const variable_list s = ctx->get_saved_variables();
        const Problem p = load(ctx);
        // a saved-tensor hook may bring a tensor back in another layout
        const std::array<Tensor, 5> in{view(s[0]), view(s[1]), view(s[2]), view(s[3]), view(s[4])};
        const Tensor& q = in[0];
        const Tensor o = s[5].contiguous(), lse = s[6].contiguous();
        const c10::OptionalDeviceGuard guard(q.device());
        const Tensor d_o = view(grad[0].scalar_type() == q.scalar_type() ? grad[0] : grad[0].to(q.scalar_type()));
        const int B = (int)q.size(0), H = (int)q.size(1), T = (int)q.size(2), D = (int)q.size(3);
        const int code = dtype_code(q.scalar_type());
        const Layouts l = layouts_of(in);
        const bool dense = l.dense && d_o.is_contiguous();
        const int w1 = (int)p.w[0], w2 = (int)p.w[1], kl = (int)p.w[2], kr = (int)p.w[3];
        const unsigned flags = (unsigned)p.flags;
        variable_list g(6);
        void* gp[5];
        for (int i = 0; i < 5; ++i) {  // only the gradients autograd asks for
            if (ctx->needs_input_grad(i)) g[i] = gradient_like(q);
            gp[i] = g[i].defined() ? g[i].data_ptr() : nullptr;
        }
        // null: that side is dense
        const tritt_layout ldo = layout_of(d_o);
        const tritt_layout *lp = l.dense ? nullptr : l.at.data(), *ldp = d_o.is_contiguous() ? nullptr : &ldo;
        const size_t need = dense ? tritt_tdp_bwd_workspace_bytes(B, H, T, D, code, p.causal, w1, w2, kl, kr, flags)
                                  : tritt_tdp_bwd_strided_workspace_bytes(B, H, T, D, code, p.causal, w1, w2, kl, kr, flags, lp,
                                                                          ldp);
        const Tensor ws = workspace(need, q);
        void* st = current_stream(q);
        check(dense ? tritt_tdp_bwd(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                    o.data_ptr(), lse.data_ptr<float>(), d_o.data_ptr(), gp[0], gp[1], gp[2], gp[3], gp[4], B,
                                    H, T, D, code, (float)p.scale, p.causal, w1, w2, kl, kr, ws.data_ptr(), ws.numel(), flags,
                                    st)
                    : tritt_tdp_bwd_strided(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(),
                                            in[4].data_ptr(), lp, o.data_ptr(), lse.data_ptr<float>(), d_o.data_ptr(), ldp,
                                            gp[0], gp[1], gp[2], gp[3], gp[4], B, H, T, D, code, (float)p.scale, p.causal, w1,
                                            w2, kl, kr, ws.data_ptr(), ws.numel(), flags, st),
              "tritt_tdp_bwd");
        return g;
    }
};

struct Dps : torch::autograd::Function<Dps> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k1_, const Tensor& k2_,
                                 const Tensor& v1_, const Tensor& v2_, const Problem& p) {
        const std::array<Tensor, 5> in{view(q_), view(k1_), view(k2_), view(v1_), view(v2_)};
        const Tensor& q = in[0];
        const c10::OptionalDeviceGuard guard(q.device());
        const int B = (int)q.size(0), H = (int)q.size(1), T = (int)q.size(2), D = (int)q.size(3);
        const int code = dtype_code(q.scalar_type()), k_diff = (int)p.w[0];
        const unsigned flags = (unsigned)p.flags;
        Tensor o = gradient_like(q), m = at::empty({B, H, T}, q.options().dtype(at::kFloat));
        const Layouts l = layouts_of(in);
        const Tensor ws = workspace(l.dense ? tritt_dps_fwd_workspace_bytes(B, H, T, D, code, flags)
                                            : tritt_dps_fwd_strided_workspace_bytes(B, H, T, D, code, flags, l.at.data()),
                                    q);
        void* st = current_stream(q);
        if (p.keep) {
            const Tensor r = at::empty({B, H, T, D}, m.options()), lse1 = at::empty({B, H, (T + 31) / 32 * 32}, m.options());
            check(tritt_dps_fwd_keep(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                     l.dense ? nullptr : l.at.data(), o.data_ptr(), m.data_ptr<float>(), r.data_ptr<float>(),
                                     lse1.data_ptr<float>(), B, H, T, D, code, (float)p.scale, p.causal, k_diff, ws.data_ptr(),
                                     ws.numel(), flags, st),
                  "tritt_dps_fwd_keep");
            ctx->save_for_backward({in[0], in[1], in[2], in[3], in[4], o, m, r, lse1});
            ctx->mark_non_differentiable({m});
            save(ctx, p);
            return {o, m};
        }
        check(l.dense ? tritt_dps_fwd(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                      o.data_ptr(), m.data_ptr<float>(), B, H, T, D, code, (float)p.scale, p.causal, k_diff,
                                      ws.data_ptr(), ws.numel(), flags, st)
                      : tritt_dps_fwd_strided(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(),
                                              in[4].data_ptr(), l.at.data(), o.data_ptr(), m.data_ptr<float>(), B, H, T, D,
                                              code, (float)p.scale, p.causal, k_diff, ws.data_ptr(), ws.numel(), flags, st),
              "tritt_dps_fwd");
        ctx->save_for_backward({in[0], in[1], in[2], in[3], in[4], o, m});
        ctx->mark_non_differentiable({m});
        save(ctx, p);
        return {o, m};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grad) {
        const variable_list s = ctx->get_saved_variables();
        const Problem p = load(ctx);
        const std::array<Tensor, 5> in{view(s[0]), view(s[1]), view(s[2]), view(s[3]), view(s[4])};
        const Tensor& q = in[0];
        const Tensor o = s[5].contiguous(), m = s[6].contiguous();
        const c10::OptionalDeviceGuard guard(q.device());
        if (grad[0].sizes() != o.sizes() || grad[0].device() != o.device() || grad[0].scalar_type() != o.scalar_type())
            throw std::runtime_error("TrittentionTriton: dO must have the shape, the device and the dtype of O");
        const Tensor d_o = view(grad[0]);
        const int B = (int)q.size(0), H = (int)q.size(1), T = (int)q.size(2), D = (int)q.size(3);
        const int code = dtype_code(q.scalar_type()), k_diff = (int)p.w[0];
        const unsigned flags = (unsigned)p.flags;
        const Layouts l = layouts_of(in);
        const bool all_dense = l.dense && d_o.is_contiguous();
        variable_list g(6);
        void* gp[5];
        for (int i = 0; i < 5; ++i) {
            g[i] = gradient_like(q);
            gp[i] = g[i].data_ptr();
        }
        const tritt_layout ldo = layout_of(d_o);
        const tritt_layout *lp = l.dense ? nullptr : l.at.data(), *ldp = d_o.is_contiguous() ? nullptr : &ldo;
        const Tensor ws = workspace(all_dense ? tritt_dps_bwd_workspace_bytes(B, H, T, D, code, flags)
                                              : tritt_dps_bwd_strided_workspace_bytes(B, H, T, D, code, flags, lp, ldp),
                                    q);
        void* st = current_stream(q);
        if (s.size() > 7) {
            const Tensor r = dense(s[7]), lse1 = dense(s[8]);
            check(tritt_dps_bwd_kept(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(), lp,
                                     o.data_ptr(), m.data_ptr<float>(), r.data_ptr<float>(), lse1.data_ptr<float>(),
                                     d_o.data_ptr(), ldp, gp[0], gp[1], gp[2], gp[3], gp[4], B, H, T, D, code, (float)p.scale,
                                     p.causal, k_diff, ws.data_ptr(), ws.numel(), flags, st),
                  "tritt_dps_bwd_kept");
            return g;
        }
        check(all_dense ? tritt_dps_bwd(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(), in[4].data_ptr(),
                                    o.data_ptr(), m.data_ptr<float>(), d_o.data_ptr(), gp[0], gp[1], gp[2], gp[3], gp[4], B, H,
                                    T, D, code, (float)p.scale, p.causal, k_diff, ws.data_ptr(), ws.numel(), flags, st)
                    : tritt_dps_bwd_strided(q.data_ptr(), in[1].data_ptr(), in[2].data_ptr(), in[3].data_ptr(),
                                            in[4].data_ptr(), lp, o.data_ptr(), m.data_ptr<float>(), d_o.data_ptr(), ldp,
                                            gp[0], gp[1], gp[2], gp[3], gp[4], B, H, T, D, code, (float)p.scale, p.causal,
                                            k_diff, ws.data_ptr(), ws.numel(), flags, st),
              "tritt_dps_bwd");
        return g;
    }
};

// ---- Python entry points -------------------------------------------------------------------------------------------------
// Whether a Python Function would see its arguments as they are: no functorch transform is active (it refuses or rewrites
// Functions, also where no argument is wrapped) and torch.jit.trace, which records a Python Function, is not recording.
bool plain_context() {
    return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !torch::jit::tracer::isTracing();
}
// the five tensors of a call in the usual case
std::optional<std::array<Tensor, 5>> usual_tensors(PyObject* const* args) {
    if (!plain_context()) return std::nullopt;
    // a GPU tensor with or without autograd; any other key (Python, functorch, Functionalize, Conjugate, Negative,
    // ZeroTensor, ...) is a wrapper or a lazy form whose storage is not the tensor
    static const c10::DispatchKeySet plain =
        c10::DispatchKeySet{c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView,
                            c10::DispatchKey::AutocastCUDA};
    std::array<Tensor, 5> t;
    for (int i = 0; i < 5; ++i) {
        if (!THPVariable_CheckExact(args[i])) return std::nullopt;
        t[i] = THPVariable_Unpack(args[i]);
        if (!t[i].is_cuda() || t[i].layout() != at::kStrided || (t[i].key_set().raw_repr() & ~plain.raw_repr()) ||
            t[i]._fw_grad(0).defined())
            return std::nullopt;
        if (t[i].dim() != 4 || dtype_code(t[i].scalar_type()) < 0) return std::nullopt;
        if (i && (t[i].sizes() != t[0].sizes() || t[i].scalar_type() != t[0].scalar_type() || t[i].device() != t[0].device()))
            return std::nullopt;
    }
    const int64_t D = t[0].size(3);
    if (D != 8 && D != 16 && D != 32 && D != 64 && D != 128) return std::nullopt;
    for (int i = 0; i < 3; ++i)
        if (t[0].size(i) > 0x7fffffff) return std::nullopt;
    return t;
}
// None or a non-negative int, clamped to the sequence length (None: no window)
bool window(PyObject* o, int64_t T, int64_t* out) {
    if (o == Py_None) {
        *out = T;
        return true;
    }
    if (!PyLong_Check(o)) return false;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow > 0) {
        *out = T;
        return true;
    }
    if (overflow < 0 || v < 0) return false;
    *out = std::min<int64_t>(v, T);
    return true;
}
bool number(PyObject* o, double* out) {
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
    *out = PyFloat_AsDouble(o);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

bool truth(PyObject* o, bool* out) {
    const int v = PyObject_IsTrue(o);
    *out = v == 1;
    if (v >= 0) return true;
    PyErr_Clear();
    return false;
}

// tdp(q, k1, k2, v1, v2, softmax_scale, kk_left, kk_right, k1_window, k2_window, causal, convert_to_float32) -> O or None
PyObject* py_tdp(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS  // torch's own exception types, and those of Python code called back (saved-tensor hooks)
        if (n != 12) {
            PyErr_SetString(PyExc_TypeError, "tdp takes 12 arguments");
            return nullptr;
        }
        auto t = usual_tensors(args);
        Problem p{};
        bool convert = false;
        if (!t || !number(args[5], &p.scale) || !truth(args[10], &p.causal) || !truth(args[11], &convert)) Py_RETURN_NONE;
        const int64_t T = (*t)[0].size(2), D = (*t)[0].size(3);
        if (!window(args[8], T, &p.w[0]) || !window(args[9], T, &p.w[1]) || !window(args[6], T, &p.w[2]) ||
            !window(args[7], T, &p.w[3]))
            Py_RETURN_NONE;
        if (convert)
            p.flags = ((*t)[0].scalar_type() != at::kFloat && (D == 32 || D == 64)) ? TRITT_FLAG_SPLIT_OPERANDS
                                                                                     : TRITT_FLAG_FORCE_GENERIC;
        Tensor o;
        {
            pybind11::gil_scoped_release release;
            o = Tdp::apply((*t)[0], (*t)[1], (*t)[2], (*t)[3], (*t)[4], p);
        }
        return THPVariable_Wrap(std::move(o));
    END_HANDLE_TH_ERRORS
}

// dps(q, k1, k2, v1, v2, causal, softmax_scale, k_diff, convert_to_float32) -> (o, m) or None
PyObject* py_dps(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
        if (n != 9) {
            PyErr_SetString(PyExc_TypeError, "dps takes 9 arguments");
            return nullptr;
        }
        auto t = usual_tensors(args);
        Problem p{};
        bool convert = false;
        if (!t || !number(args[6], &p.scale) || !window(args[7], (*t)[0].size(2), &p.w[0]) || !truth(args[5], &p.causal) ||
            !truth(args[8], &convert))
            Py_RETURN_NONE;
        if (convert) p.flags = TRITT_FLAG_FORCE_GENERIC;
        if (at::GradMode::is_enabled() && tritt_dps_keeps((int)(*t)[0].size(3), dtype_code((*t)[0].scalar_type()), (unsigned)p.flags))
            for (const Tensor& x : *t) p.keep = p.keep || x.requires_grad();
        variable_list r;
        {
            pybind11::gil_scoped_release release;
            r = Dps::apply((*t)[0], (*t)[1], (*t)[2], (*t)[3], (*t)[4], p);
        }
        PyObject* pair = PyTuple_New(2);
        if (!pair) return nullptr;
        for (int i = 0; i < 2; ++i) PyTuple_SET_ITEM(pair, i, THPVariable_Wrap(std::move(r[i])));
        return pair;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"tdp", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_tdp)), METH_FASTCALL,
     "Triple-dot attention with autograd in native code; None where the Python Function has to decide."},
    {"dps", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_dps)), METH_FASTCALL,
     "Dot-product-sum attention with autograd in native code; None where the Python Function has to decide."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "torch tensors to the C ABI of libtrittention_hip.so", -1, methods};

}  // namespace

// torch_version: what this was compiled against; torch's C++ interfaces change from one version to the next
PyMODINIT_FUNC PyInit__native(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
