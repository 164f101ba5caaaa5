// race_torch.cpp -- the autograd calls of race_attention_amd.functional as C++
// autograd Functions over the C ABI (include/race_attention.h).
//
// A call of the operator is two or three kernels each way, 10 to 30 us at a few
// thousand tokens, while the Python path -- descriptor, size queries, six
// allocations, ctypes calls, a Python autograd node in each direction -- takes
// 40 us forward and 150 us with its backward, and the learnable temperature's
// exp, clamp and reciprocal with their backward another 150 us and 15 launches.
// Here a call costs its checks, allocations and launches, the backward runs in
// the engine's thread without the interpreter, and the temperature is one launch
// each way (race_inv_temp).
//
// These functions take the ordinary calls: plain CUDA tensors on the current
// device, bf16 or fp32, shapes and arguments that agree.  For everything else
// (mismatched shapes, CPU tensors, tensor subclasses, functorch transforms,
// tracing, an active dispatch mode, a status other than RACE_OK) they return None and the caller takes the
// Python path, whose errors and conversions are then what they always were.
#include <dlfcn.h>
#include <torch/extension.h>

#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <string>

#include "../../include/race_attention.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------ the operator library
#define RACE_FNS(X)                                                                                              \
    X(race_state_bytes) X(race_fwd_workspace_bytes) X(race_bwd_workspace_bytes) X(race_fwd) X(race_bwd)          \
    X(race_fwd_ex_workspace_bytes) X(race_fwd_ex) X(race_bwd_ex) X(race_fwd_padded) X(race_bwd_padded)           \
    X(race_fwd_global_workspace_bytes)                                                                            \
    X(race_bwd_global_workspace_bytes) X(race_fwd_global) X(race_bwd_global) X(race_probs_bwd_workspace_bytes)   \
    X(race_probs) X(race_probs_bwd) X(race_inv_temp) X(race_last_error)
struct Lib {
#define X(f) decltype(&::f) f = nullptr;
    RACE_FNS(X)
#undef X
} lib;
PyObject *race_error = nullptr;  // _lib.RaceError

// The library that ctypes loaded (the same file: the same handle).
void bind(const std::string &path, py::object error) {
    void *h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(h, "cannot load ", path, ": ", dlerror());
    Lib l;
#define X(f)                                                        \
    l.f = reinterpret_cast<decltype(&::f)>(dlsym(h, #f));           \
    TORCH_CHECK(l.f, path, " does not export ", #f);
    RACE_FNS(X)
#undef X
    lib = l;
    race_error = error.release().ptr();
}

// A call that these functions do not take, or whose status is an error.
struct NotTaken {};

[[noreturn]] void raise_status(const char *what, int rc) {
    const std::string msg = std::string(what) + " failed (" + std::to_string(rc) + "): " + lib.race_last_error();
    py::gil_scoped_acquire gil;
    PyErr_SetString(race_error, msg.c_str());
    python_error e;
    e.persist();
    throw e;
}

// ------------------------------------------------------------ arguments
void *stream_of(const Tensor &x) { return (void *)c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

// a plain strided CUDA tensor of the current device: no wrapper of a transform, a mode or a subclass
bool plain(const Tensor &x) {
    return x.defined() && x.is_cuda() && x.layout() == at::kStrided && x.unsafeGetTensorImpl()->has_storage() &&
           !x.unsafeGetTensorImpl()->is_python_dispatch() && !x.is_conj() && !x.is_neg() &&
           !x._fw_grad(/*level=*/0).defined();  // forward-mode AD: refused by the Python Functions
}
// torch.Tensor or torch.nn.Parameter itself (THPVariable_CheckExact takes both), no other subclass
bool is_tensor(py::handle o) { return THPVariable_CheckExact(o.ptr()); }

bool aligned(const Tensor &x) {
    const int64_t es = x.element_size();
    if (x.stride(4) != 1 || reinterpret_cast<uintptr_t>(x.data_ptr()) % 16) return false;
    for (int j = 0; j < 4; ++j)
        if (x.size(j) != 1 && (x.stride(j) * es) % 16) return false;
    return x.size(2) == 1 || x.stride(2) >= x.size(4);
}
// usable by the kernels: contiguous D, 16-byte aligned rows
Tensor usable(const Tensor &x) { return aligned(x) ? x : x.contiguous(); }
void strides4(const Tensor &x, int64_t *st) {
    for (int j = 0; j < 4; ++j) st[j] = x.size(j) > 1 ? x.stride(j) : 0;
}
void *ptr(const Tensor &x) { return x.data_ptr(); }
float *fptr(const Tensor &x) { return x.defined() ? static_cast<float *>(x.data_ptr()) : nullptr; }

enum Kind : int64_t { F1 = 0, EX = 1, GLOBAL = 2, PROBS = 3, PADDED = 4 };

// What the forward and the backward of one call share beside tensors.
struct Cfg {
    int64_t kind, L, K, causal, den;
    double eps, it, lo, hi;  // it: a host temperature; lo, hi: bounds of exp(logit), lo < 0 without a logit
    c10::IValue pack() const {
        return c10::ivalue::Tuple::create({kind, L, K, causal, den, eps, it, lo, hi});
    }
    static Cfg unpack(const c10::IValue &v) {
        const auto &e = v.toTupleRef().elements();
        return Cfg{e[0].toInt(),    e[1].toInt(),    e[2].toInt(),    e[3].toInt(),   e[4].toInt(),
                   e[5].toDouble(), e[6].toDouble(), e[7].toDouble(), e[8].toDouble()};
    }
};

void fill_desc(race_desc &d, const Cfg &c, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &planes,
               const Tensor &temp) {
    memset(&d, 0, sizeof d);
    d.M = q.size(0);
    d.B = q.size(1);
    d.T = q.size(2);
    d.H = q.size(3);
    d.D = q.size(4);
    d.L = (int32_t)c.L;
    d.K = (int32_t)c.K;
    d.causal = (int32_t)c.causal;
    d.dtype = q.scalar_type() == at::kBFloat16 ? RACE_DTYPE_BF16 : RACE_DTYPE_F32;
    d.eps = (float)c.eps;
    d.inv_temp = temp.defined() ? 1.f : (float)c.it;
    d.inv_temp_ptr = temp.defined() ? fptr(temp) : nullptr;
    d.planes_m_stride = planes.dim() == 4 && planes.size(0) > 1 ? c.L * c.K * d.D : 0;
    strides4(q, d.q_stride);
    strides4(k, d.k_stride);
    strides4(v, d.v_stride);
}

Tensor bytes(size_t n, const Tensor &like) {
    return at::empty({(int64_t)(n < 16 ? 16 : n)}, like.options().dtype(at::kByte));
}
Tensor fp32(at::IntArrayRef shape, const Tensor &like) { return at::empty(shape, like.options().dtype(at::kFloat)); }

// The temperature a call runs with: a device copy (made now: the source may be
// updated in place before the backward), or for a logit the pair (inv_temp,
// d inv_temp / d logit).  Undefined for a host temperature.
Tensor device_temp(const Cfg &c, const Tensor &temp, const Tensor &q) {
    if (!temp.defined()) return Tensor();
    if (c.lo >= 0) {
        Tensor t = fp32({2}, q);
        if (lib.race_inv_temp(fptr(temp), (float)c.lo, (float)c.hi, fptr(t), stream_of(q)) != RACE_OK) throw NotTaken();
        return t;
    }
    return temp.detach().to(at::kFloat).clone();
}

struct Fwd {
    Tensor out, den, state, temp;
};
Fwd forward_impl(const Cfg &c, const Tensor &q0, const Tensor &k0, const Tensor &v0, const Tensor &planes,
                 const Tensor &temp, const Tensor &kmask) {
    const Tensor q = usable(q0), k = usable(k0), v = usable(v0);
    Fwd f;
    f.temp = device_temp(c, temp, q);
    race_desc d;
    fill_desc(d, c, q, k, v, planes, f.temp);
    f.out = at::empty(q0.sizes(), q.options());
    strides4(f.out, d.o_stride);
    const size_t sb = lib.race_state_bytes(&d);
    if (!sb) throw NotTaken();
    f.state = bytes(sb, q);
    if (c.den) f.den = fp32({d.M, d.B, d.H, d.T}, q);
    const bool ex = c.kind == EX || c.kind == PADDED;
    const Tensor ws = bytes(c.kind == F1 ? lib.race_fwd_workspace_bytes(&d)
                            : ex         ? lib.race_fwd_ex_workspace_bytes(&d)
                                         : lib.race_fwd_global_workspace_bytes(&d),
                            q);
    void *s = stream_of(q);
    const size_t wb = (size_t)ws.numel();
    const int rc =
        c.kind == F1 ? lib.race_fwd(&d, ptr(q), ptr(k), ptr(v), fptr(planes), ptr(f.out), ptr(f.state), ptr(ws), wb, s)
        : ex
            ? (c.kind == EX ? lib.race_fwd_ex : lib.race_fwd_padded)(&d, ptr(q), ptr(k), ptr(v), fptr(planes),
                                                                     fptr(kmask), ptr(f.out), fptr(f.den),
                                                                     ptr(f.state), ptr(ws), wb, s)
            : lib.race_fwd_global(&d, ptr(q), ptr(k), ptr(v), fptr(planes), ptr(f.out), fptr(f.den), ptr(f.state),
                                  ptr(ws), wb, s);
    if (rc != RACE_OK) throw NotTaken();
    return f;
}

// d(inv_temp), or through a logit's exp, clamp and reciprocal, in the type of the source
Tensor temp_grad(const Cfg &c, const Tensor &git, const Tensor &temp, at::ScalarType type) {
    return (c.lo >= 0 ? at::mul(git, temp.select(0, 1)) : git).to(type);
}

struct Operator : torch::autograd::Function<Operator> {
    static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                                 const Tensor &planes, const std::optional<Tensor> &otemp,
                                 const std::optional<Tensor> &okmask, c10::IValue cfg) {
        const Cfg c = Cfg::unpack(cfg);
        const Tensor temp = otemp.value_or(Tensor()), kmask = okmask.value_or(Tensor());
        const Fwd f = forward_impl(c, q, k, v, planes, temp, kmask);
        ctx->set_materialize_grads(c.kind == F1);
        ctx->saved_data["cfg"] = cfg;
        if (temp.defined()) ctx->saved_data["type"] = (int64_t)temp.scalar_type();
        const bool gl = c.kind == GLOBAL;
        ctx->save_for_backward({q, k, v, planes, kmask, f.state, f.temp, gl ? f.out : Tensor(), gl ? f.den : Tensor()});
        return c.den ? variable_list{f.out, f.den} : variable_list{f.out};
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &planes = saved[3], &kmask = saved[4], &state = saved[5], &temp = saved[6];
        const Cfg c = Cfg::unpack(ctx->saved_data["cfg"]);
        const Tensor q = usable(saved[0]), k = usable(saved[1]), v = usable(saved[2]);
        const Tensor dout =
            grads[0].defined() ? usable(grads[0].to(q.scalar_type())) : at::zeros(saved[0].sizes(), q.options());
        Tensor dden = grads.size() > 1 ? grads[1] : Tensor();
        if (dden.defined()) dden = dden.to(at::kFloat).contiguous();
        race_desc d;
        fill_desc(d, c, q, k, v, planes, temp);
        strides4(dout, d.do_stride);
        const Tensor dq = at::empty(saved[0].sizes(), q.options()), dk = at::empty_like(dq), dv = at::empty_like(dq);
        strides4(dq, d.g_stride);
        const bool want = temp.defined() && ctx->needs_input_grad(4);  // (an absent temperature is no edge)
        const Tensor git = want ? fp32({}, q) : Tensor();
        const Tensor ws = bytes(c.kind == GLOBAL ? lib.race_bwd_global_workspace_bytes(&d)
                                                 : lib.race_bwd_workspace_bytes(&d), q);
        void *s = stream_of(q);
        const size_t wb = (size_t)ws.numel();
        int rc;
        if (c.kind == F1) {
            rc = lib.race_bwd(&d, ptr(q), ptr(k), ptr(v), fptr(planes), ptr(dout), ptr(state), ptr(dq), ptr(dk),
                              ptr(dv), fptr(git), ptr(ws), wb, s);
        } else if (c.kind == EX || c.kind == PADDED) {
            rc = (c.kind == EX ? lib.race_bwd_ex : lib.race_bwd_padded)(
                &d, ptr(q), ptr(k), ptr(v), fptr(planes), fptr(kmask), ptr(dout), fptr(dden), ptr(state), ptr(dq),
                ptr(dk), ptr(dv), fptr(git), ptr(ws), wb, s);
        } else {
            const Tensor out = usable(saved[7]);
            strides4(out, d.o_stride);
            rc = lib.race_bwd_global(&d, ptr(q), ptr(k), ptr(v), fptr(planes), ptr(out), fptr(saved[8]), ptr(dout),
                                     fptr(dden), ptr(state), ptr(dq), ptr(dk), ptr(dv), fptr(git), ptr(ws), wb, s);
        }
        if (rc != RACE_OK) raise_status("race_bwd", rc);
        Tensor dt;
        if (want) dt = temp_grad(c, git, temp, (at::ScalarType)ctx->saved_data["type"].toInt());
        return {ctx->needs_input_grad(0) ? dq : Tensor(), ctx->needs_input_grad(1) ? dk : Tensor(),
                ctx->needs_input_grad(2) ? dv : Tensor(), Tensor(), dt, Tensor(), Tensor()};
    }
};

Tensor probs_impl(const Cfg &c, const Tensor &x0, const Tensor &planes, const Tensor &temp) {
    const Tensor x = usable(x0);
    race_desc d;
    fill_desc(d, c, x, x, x, planes, temp);
    const Tensor P = fp32({d.M, d.B, d.H, d.T, c.L << c.K}, x);
    if (lib.race_probs(&d, ptr(x), fptr(planes), fptr(P), stream_of(x)) != RACE_OK) throw NotTaken();
    return P;
}

struct Probs : torch::autograd::Function<Probs> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &planes,
                          const std::optional<Tensor> &otemp, c10::IValue cfg) {
        const Cfg c = Cfg::unpack(cfg);
        const Tensor temp = otemp.value_or(Tensor());
        const Tensor t = device_temp(c, temp, x);
        const Tensor P = probs_impl(c, x, planes, t);
        ctx->saved_data["cfg"] = cfg;
        if (temp.defined()) ctx->saved_data["type"] = (int64_t)temp.scalar_type();
        ctx->save_for_backward({x, planes, t});
        return P;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Cfg c = Cfg::unpack(ctx->saved_data["cfg"]);
        const Tensor x = usable(saved[0]), &planes = saved[1], &temp = saved[2];
        const Tensor dP = grads[0].to(at::kFloat).contiguous();
        race_desc d;
        fill_desc(d, c, x, x, x, planes, temp);
        const Tensor dx = at::empty(saved[0].sizes(), x.options());
        strides4(dx, d.g_stride);
        const bool want = temp.defined() && ctx->needs_input_grad(2);
        const Tensor git = want ? fp32({}, x) : Tensor();
        const Tensor ws = bytes(lib.race_probs_bwd_workspace_bytes(&d), x);
        const int rc = lib.race_probs_bwd(&d, ptr(x), fptr(planes), fptr(dP), ptr(dx), fptr(git), ptr(ws),
                                          (size_t)ws.numel(), stream_of(x));
        if (rc != RACE_OK) raise_status("race_probs_bwd", rc);
        Tensor dt;
        if (want) dt = temp_grad(c, git, temp, (at::ScalarType)ctx->saved_data["type"].toInt());
        return {ctx->needs_input_grad(0) ? dx : Tensor(), Tensor(), dt, Tensor()};
    }
};

std::optional<Tensor> given(const Tensor &x) { return x.defined() ? std::optional<Tensor>(x) : std::nullopt; }

// ------------------------------------------------------------ Python entry
// q, k, v: one input tensor of each (probabilities: x three times); planes
// [L,K,D], [1,L,K,D] or [M,L,K,D]; temp: a float, a CUDA tensor, or with lo >= 0
// the logit of an fp32 temperature clamped to [lo, hi].
py::object call(int64_t kind, py::handle hq, py::handle hk, py::handle hv, py::handle hplanes, py::handle htemp,
                py::handle hmask, int64_t L, int64_t K, bool causal, bool want_den, double eps, double lo, double hi) {
    if (!is_tensor(hq) || !is_tensor(hk) || !is_tensor(hv) || !is_tensor(hplanes) || torch::jit::tracer::isTracing() ||
        c10::impl::TorchDispatchModeTLS::any_modes_set())
        return py::none();
    const Tensor &q = THPVariable_Unpack(hq.ptr()), &k = THPVariable_Unpack(hk.ptr()), &v = THPVariable_Unpack(hv.ptr());
    Tensor planes = THPVariable_Unpack(hplanes.ptr()), temp, mask;
    if (!plain(q) || !plain(k) || !plain(v) || !plain(planes) || q.device().index() != c10::hip::current_device()) return py::none();
    if (q.dim() != 5 || k.sizes() != q.sizes() || v.sizes() != q.sizes() || q.numel() == 0 ||
        k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || k.device() != q.device() ||
        v.device() != q.device() || (q.scalar_type() != at::kBFloat16 && q.scalar_type() != at::kFloat))
        return py::none();
    if (q.stride(4) != 1 || k.stride(4) != 1 || v.stride(4) != 1) return py::none();
    const int64_t pd = planes.dim();
    if ((pd != 3 && pd != 4) || planes.size(pd - 3) != L || planes.size(pd - 2) != K || planes.size(pd - 1) != q.size(4) ||
        (pd == 4 && planes.size(0) != 1 && planes.size(0) != q.size(0)))
        return py::none();
    Cfg c{kind, L, K, causal, want_den, eps, 0.0, -1.0, 0.0};
    if (PyFloat_Check(htemp.ptr())) {
        c.it = PyFloat_AS_DOUBLE(htemp.ptr());
    } else {
        if (!is_tensor(htemp)) return py::none();
        temp = THPVariable_Unpack(htemp.ptr());
        if (!plain(temp) || temp.device() != q.device() || temp.dim() != 0 || !at::isFloatingType(temp.scalar_type()))
            return py::none();
        if (lo >= 0) {
            if (temp.scalar_type() != at::kFloat) return py::none();
            c.lo = lo;
            c.hi = hi;
        }
    }
    if (!hmask.is_none()) {
        if (!is_tensor(hmask)) return py::none();
        mask = THPVariable_Unpack(hmask.ptr());
        if (!plain(mask) || mask.requires_grad() || mask.dim() != 2 || mask.size(0) != q.size(1) || mask.size(1) != q.size(2)) return py::none();
    }
    if (kind == PADDED && !mask.defined()) return py::none();
    try {
        py::gil_scoped_release nogil;
        const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad() ||
                                                         (temp.defined() && temp.requires_grad()));
        {
            at::NoGradGuard ng;  // buffers: no gradient
            planes = planes.to(q.device(), at::kFloat).contiguous();
            if (mask.defined()) mask = mask.to(q.device(), at::kFloat).contiguous();
        }
        if (kind == PROBS) {
            const Tensor P = grad ? Probs::apply(q, planes, given(temp), c.pack())
                                  : probs_impl(c, q.detach(), planes, device_temp(c, temp.defined() ? temp.detach() : temp, q));
            py::gil_scoped_acquire gil;
            return py::cast(P);
        }
        variable_list r;
        if (grad) {
            r = Operator::apply(q, k, v, planes, given(temp), given(mask), c.pack());
        } else {
            const Fwd f = forward_impl(c, q.detach(), k.detach(), v.detach(), planes,
                                       temp.defined() ? temp.detach() : temp, mask);
            r = c.den ? variable_list{f.out, f.den} : variable_list{f.out};
        }
        py::gil_scoped_acquire gil;
        return r.size() == 1 ? py::cast(r[0]) : py::object(py::make_tuple(r[0], r[1]));
    } catch (const NotTaken &) {
        return py::none();
    }
}

} // namespace

PYBIND11_MODULE(_race_torch, m) {
    m.def("bind", &bind);
    m.def("call", &call);
    m.attr("F1") = (int64_t)F1;
    m.attr("EX") = (int64_t)EX;
    m.attr("GLOBAL") = (int64_t)GLOBAL;
    m.attr("PROBS") = (int64_t)PROBS;
    m.attr("PADDED") = (int64_t)PADDED;
}
