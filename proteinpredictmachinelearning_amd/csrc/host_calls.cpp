// The operators of ops.py for ordinary arguments, from Python's call to the launcher in one piece of native code.
//
// What bounds a small call is the host: a projection of 408 x 256 -> 256, whose kernel takes 4.0 us, cost 6.4 through ops.py and
// ctypes -- 2.7 the launch, 1.4 torch.empty, 0.6 the ctypes call, the rest the checks of its arguments -- and 4.2 through this
// module, the kernel's own time.  2601 x 128 -> 132 6.7 -> 5.2, 1672 x 64 -> 192 on a Q8_0 weight 6.5 -> 4.5.
//
// A function here takes a call only if everything about it is ordinary: plain torch.Tensors (no subclass, no transform's or mode's
// wrapper, no active mode), on the current device, which ppml_hip_init has seen, of the expected type, contiguous, of matching sizes,
// on the default stream.  Anything else, and any launcher that does not return 0, is answered with None: ops.py then does the call its long
// way, which is where errors are worded.  No state is kept but the launchers' addresses and the devices that are ready.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cstdint>
#include <cstring>

namespace {

enum Launcher { MUL_MAT, MUL_MAT_F16, MUL_MAT_Q8, MUL_MAT_Q8_EX, OPM, OPM_BACK, TRI_MUL, TRI_MUL_BACK, ATTN, ATTN_BACK, LAUNCHERS };
const char* const LAUNCHER_NAMES[LAUNCHERS] = {"mul_mat_hip", "mul_mat_f16_hip", "mul_mat_q8_hip", "mul_mat_q8_ex_hip", "outer_prod_mean_hip", "outer_prod_mean_back_hip",
                                               "tri_mul_hip", "tri_mul_back_hip", "flash_attn_forward_ex_hip", "flash_attn_backward_hip"};
void* g_launcher[LAUNCHERS];
std::atomic<uint64_t> g_ready{0};                       // a bit per device

using at::Tensor;

struct Call {
    c10::Device device{c10::DeviceType::CPU};
    bool ordinary = true;

    // the default stream of a device that is ready, and nobody listening
    Call() {
        const c10::impl::VirtualGuardImpl guard(c10::DeviceType::CUDA);
        device = guard.getDevice();
        const int i = device.index();
        ordinary = i >= 0 && i < 64 && (g_ready.load(std::memory_order_acquire) >> i & 1) != 0 && guard.getStream(device).id() == 0 &&
                   !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set();
    }
    // `obj` as a tensor of this call (a null pointer for None where that is allowed)
    const Tensor* tensor(PyObject* obj, at::ScalarType type, bool optional = false) {
        static const c10::DispatchKeySet plain({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
        if (!ordinary || (optional && obj == Py_None)) return nullptr;
        if (!THPVariable_CheckExact(obj)) { ordinary = false; return nullptr; }
        const Tensor& t = THPVariable_Unpack(obj);
        ordinary = t.defined() && (t.key_set().raw_repr() & ~plain.raw_repr()) == 0 && t.layout() == at::kStrided && t.scalar_type() == type && t.device() == device &&
                   t.is_contiguous() && !t.is_conj() && !t.is_neg();
        return ordinary ? &t : nullptr;
    }
    Tensor empty(at::IntArrayRef sizes) const { return at::empty(sizes, at::TensorOptions().dtype(at::kFloat).device(device)); }
};

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject* wrap_or_none(Tensor t) { return t.defined() ? THPVariable_Wrap(std::move(t)) : none(); }
float* f(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }
const float* f(const Tensor* t) { return t ? static_cast<const float*>(t->const_data_ptr()) : nullptr; }
bool fits(int64_t x) { return x >= 0 && x <= 0x7fffffff; }

template <class... Args>
int launch(Launcher which, Args... args) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = reinterpret_cast<int (*)(Args...)>(g_launcher[which])(args...);
    Py_END_ALLOW_THREADS
    return rc;
}

// C++ exceptions (an allocation that fails) end here: the long way meets them again and says so
template <class Body>
PyObject* guarded(Body body) {
    try {
        return body();
    } catch (...) {
        PyErr_Clear();
        return none();
    }
}

bool integer(PyObject* obj, int64_t& out) {
    if (!PyLong_CheckExact(obj) && !PyBool_Check(obj)) return false;
    int overflow = 0;
    out = PyLong_AsLongLongAndOverflow(obj, &overflow);
    return overflow == 0;
}
bool number(PyObject* obj, double& out) {
    if (PyFloat_CheckExact(obj)) { out = PyFloat_AS_DOUBLE(obj); return true; }
    int64_t i;
    if (!integer(obj, i) || i > (1LL << 53) || i < -(1LL << 53)) return false;
    out = static_cast<double>(i);
    return true;
}

typedef const float* cf;
typedef const void* cv;

// (a, b, bias)
template <Launcher which>
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (n != 3) return none();
        Call call;
        const at::ScalarType type = which == MUL_MAT ? at::kFloat : at::kHalf;
        const Tensor *a = call.tensor(args[0], type), *b = call.tensor(args[1], type), *bias = call.tensor(args[2], at::kFloat, true);
        if (!call.ordinary || a->dim() != 2 || b->dim() != 2 || a->size(1) != b->size(1) || (bias && bias->numel() != b->size(0))) return none();
        const int64_t M = a->size(0), K = a->size(1), N = b->size(0);
        if (M <= 0 || K <= 0 || N <= 0 || !fits(M) || !fits(K) || !fits(N)) return none();
        Tensor out = call.empty({M, N});
        const int rc = launch<cv, cv, float*, int, int, int, cf, void*>(which, a->const_data_ptr(), b->const_data_ptr(), f(out), static_cast<int>(M),
                                                                       static_cast<int>(K), static_cast<int>(N), f(bias), nullptr);
        return rc == 0 ? wrap(std::move(out)) : none();
    });
}

// (weight bytes, x, M, K, wtype, c_trans, flags)
PyObject* mul_mat_q8(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t M, K, wtype, c_trans, flags;
        if (n != 7 || !integer(args[2], M) || !integer(args[3], K) || !integer(args[4], wtype) || !integer(args[5], c_trans) || !integer(args[6], flags)) return none();
        Call call;
        const Tensor *w = call.tensor(args[0], at::kByte), *x = call.tensor(args[1], at::kFloat);
        if (!call.ordinary || x->dim() != 2 || x->size(1) != K || M <= 0 || K <= 0 || x->size(0) <= 0 || !fits(M) || !fits(K) || !fits(x->size(0)) || !fits(flags)) return none();
        const int64_t N = x->size(0);
        Tensor out = c_trans ? call.empty({N, M}) : call.empty({M, N});
        const int m = static_cast<int>(M), t = static_cast<int>(N), k = static_cast<int>(K), wt = static_cast<int>(wtype), ct = c_trans ? 1 : 0;
        const int rc = flags == 0 ? launch<cv, cf, float*, int, int, int, int, int, int*, void*>(MUL_MAT_Q8, w->const_data_ptr(), f(x), f(out), m, t, k, wt, ct, nullptr, nullptr)
                                  : launch<cv, cf, float*, int, int, int, int, int, int, void*, int32_t*, void*>(MUL_MAT_Q8_EX, w->const_data_ptr(), f(x), f(out), m, t, k, wt, ct,
                                                                                                                static_cast<int>(flags), nullptr, nullptr, nullptr);
        return rc == 0 ? wrap(std::move(out)) : none();
    });
}

// four sizes below 2^31 whose product stays below 2^62; false otherwise
bool sizes4(PyObject* const* args, int64_t (&s)[4]) {
    double product = 1.0;
    for (int i = 0; i < 4; ++i) {
        if (!integer(args[i], s[i]) || s[i] <= 0 || !fits(s[i])) return false;
        product *= static_cast<double>(s[i]);
    }
    return product < 4e18;
}

// (left, right, D, L, N, B)
PyObject* outer_product_mean(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t s[4];
        if (n != 6 || !sizes4(args + 2, s)) return none();
        const int64_t D = s[0], L = s[1], N = s[2], B = s[3];
        Call call;
        const Tensor *l = call.tensor(args[0], at::kFloat), *r = call.tensor(args[1], at::kFloat);
        if (!call.ordinary || l->numel() != D * L * N * B || r->numel() != l->numel() || static_cast<double>(D) * D * L * L * B > 4e18) return none();
        Tensor out = call.empty({D * D * L * L * B});
        const int rc = launch<cf, cf, float*, int64_t, int64_t, int64_t, int64_t, float, void*>(OPM, f(l), f(r), f(out), D, L, N, B, static_cast<float>(1.0 / static_cast<double>(N)), nullptr);
        return rc == 0 ? wrap(std::move(out)) : none();
    });
}

// (grad, left, right, D, L, N, B): both gradients
PyObject* outer_prod_mean_back(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t s[4];
        if (n != 7 || !sizes4(args + 3, s)) return none();
        const int64_t D = s[0], L = s[1], N = s[2], B = s[3];
        Call call;
        const Tensor *g = call.tensor(args[0], at::kFloat), *l = call.tensor(args[1], at::kFloat), *r = call.tensor(args[2], at::kFloat);
        if (!call.ordinary || static_cast<double>(D) * D * L * L * B > 4e18 || g->numel() != D * D * L * L * B || l->numel() != D * L * N * B || r->numel() != l->numel()) return none();
        Tensor gl = call.empty({D * L * N * B}), gr = call.empty({D * L * N * B});
        const int rc = launch<cf, cf, cf, float*, float*, int64_t, int64_t, int64_t, int64_t, float, void*>(OPM_BACK, f(g), f(l), f(r), f(gl), f(gr), D, L, N, B,
                                                                                                          static_cast<float>(1.0 / static_cast<double>(N)), nullptr);
        return rc == 0 ? Py_BuildValue("(NN)", wrap(std::move(gl)), wrap(std::move(gr))) : none();
    });
}

// (left, right, D, I, J, K, B, L, outgoing)
PyObject* tri_mul(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t s[4], B, outgoing;
        double L;
        if (n != 9 || !sizes4(args + 2, s) || !integer(args[6], B) || B <= 0 || !fits(B) || !number(args[7], L) || L == 0.0 || !integer(args[8], outgoing)) return none();
        const int64_t D = s[0], I = s[1], J = s[2], K = s[3];
        if (static_cast<double>(D) * B * I * J > 4e18 || static_cast<double>(D) * B * I * K > 4e18 || static_cast<double>(D) * B * J * K > 4e18) return none();
        Call call;
        const Tensor *l = call.tensor(args[0], at::kFloat), *r = call.tensor(args[1], at::kFloat);
        if (!call.ordinary || l->numel() != D * I * K * B || r->numel() != D * J * K * B) return none();
        Tensor out = call.empty({D * I * J * B});
        const int rc = launch<cf, cf, float*, int64_t, int64_t, int64_t, int64_t, int64_t, float, int, void*>(TRI_MUL, f(l), f(r), f(out), D, I, J, K, B, static_cast<float>(1.0 / L),
                                                                                                             outgoing ? 1 : 0, nullptr);
        return rc == 0 ? wrap(std::move(out)) : none();
    });
}

// (grad, left, right, D, I, J, K, B, L, outgoing): both gradients
PyObject* tri_mul_back(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t s[4], B, outgoing;
        double L;
        if (n != 10 || !sizes4(args + 3, s) || !integer(args[7], B) || B <= 0 || !fits(B) || !number(args[8], L) || L == 0.0 || !integer(args[9], outgoing)) return none();
        const int64_t D = s[0], I = s[1], J = s[2], K = s[3];
        if (static_cast<double>(D) * B * I * J > 4e18 || static_cast<double>(D) * B * I * K > 4e18 || static_cast<double>(D) * B * J * K > 4e18) return none();
        Call call;
        const Tensor *g = call.tensor(args[0], at::kFloat), *l = call.tensor(args[1], at::kFloat), *r = call.tensor(args[2], at::kFloat);
        if (!call.ordinary || g->numel() != D * I * J * B || l->numel() != D * I * K * B || r->numel() != D * J * K * B) return none();
        Tensor gl = call.empty({D * I * K * B}), gr = call.empty({D * J * K * B});
        const int rc = launch<cf, cf, cf, float*, float*, int64_t, int64_t, int64_t, int64_t, int64_t, float, int, void*>(
            TRI_MUL_BACK, f(g), f(l), f(r), f(gl), f(gr), D, I, J, K, B, static_cast<float>(1.0 / L), outgoing ? 1 : 0, nullptr);
        return rc == 0 ? Py_BuildValue("(NN)", wrap(std::move(gl)), wrap(std::move(gr))) : none();
    });
}

// (q, k, v, bias, causal, scale, eps, Bc, want_lse), (B, h, L, d) in and out
PyObject* flash_attn_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t causal, Bc, want_lse;
        double scale, eps;
        if (n != 9 || !integer(args[4], causal) || !number(args[5], scale) || !number(args[6], eps) || !integer(args[7], Bc) || !fits(Bc) || !integer(args[8], want_lse)) return none();
        Call call;
        const Tensor *q = call.tensor(args[0], at::kFloat), *k = call.tensor(args[1], at::kFloat), *v = call.tensor(args[2], at::kFloat),
                     *bias = call.tensor(args[3], at::kFloat, true);
        if (!call.ordinary || q->dim() != 4 || q->sizes() != k->sizes() || q->sizes() != v->sizes() || q->numel() == 0) return none();
        const int64_t B = q->size(0), h = q->size(1), L = q->size(2), d = q->size(3);
        if (!fits(B) || !fits(h) || !fits(L) || !fits(d) || (bias && bias->sizes() != at::IntArrayRef({B, h, L, L}))) return none();
        Tensor o = call.empty(q->sizes()), lse = want_lse ? call.empty({B, h, L}) : Tensor();
        const int rc = launch<int, int, int, int, int, float, float, int, cf, cf, cf, cf, float*, float*, int, void*>(
            ATTN, static_cast<int>(B), static_cast<int>(h), static_cast<int>(L), static_cast<int>(d), causal ? 1 : 0, static_cast<float>(scale), static_cast<float>(eps),
            static_cast<int>(Bc), f(q), f(k), f(v), f(bias), f(o), f(lse), 0, nullptr);
        return rc == 0 ? Py_BuildValue("(NN)", wrap(std::move(o)), wrap_or_none(std::move(lse))) : none();
    });
}

// (q, k, v, bias, o, do, lse, causal, scale, which gradients: bits dq, dk, dv, dbias)
PyObject* flash_attn_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t causal, which;
        double scale;
        if (n != 10 || !integer(args[7], causal) || !number(args[8], scale) || !integer(args[9], which) || which <= 0) return none();
        Call call;
        const Tensor *q = call.tensor(args[0], at::kFloat), *k = call.tensor(args[1], at::kFloat), *v = call.tensor(args[2], at::kFloat),
                     *bias = call.tensor(args[3], at::kFloat, true), *o = call.tensor(args[4], at::kFloat), *dout = call.tensor(args[5], at::kFloat),
                     *lse = call.tensor(args[6], at::kFloat);
        if (!call.ordinary || q->dim() != 4 || q->numel() == 0) return none();
        const int64_t B = q->size(0), h = q->size(1), L = q->size(2), d = q->size(3);
        if (!fits(B) || !fits(h) || !fits(L) || !fits(d) || k->sizes() != q->sizes() || v->sizes() != q->sizes() || o->sizes() != q->sizes() || dout->sizes() != q->sizes() ||
            lse->numel() != B * h * L || (bias && bias->numel() != B * h * L * L)) return none();
        Tensor dq, dk, dv, db;
        if (which & 1) dq = call.empty(q->sizes());
        if (which & 2) dk = call.empty(q->sizes());
        if (which & 4) dv = call.empty(q->sizes());
        if (which & 8) db = call.empty({B, h, L, L});
        const int rc = launch<int, int, int, int, int, float, cf, cf, cf, cf, cf, cf, cf, float*, float*, float*, float*, void*>(
            ATTN_BACK, static_cast<int>(B), static_cast<int>(h), static_cast<int>(L), static_cast<int>(d), causal ? 1 : 0, static_cast<float>(scale), f(q), f(k), f(v), f(bias), f(o),
            f(dout), f(lse), f(dq), f(dk), f(dv), f(db), nullptr);
        return rc == 0 ? Py_BuildValue("(NNNN)", wrap_or_none(std::move(dq)), wrap_or_none(std::move(dk)), wrap_or_none(std::move(dv)), wrap_or_none(std::move(db))) : none();
    });
}

// (name, address)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 2) { PyErr_SetString(PyExc_TypeError, "bind(name, address)"); return nullptr; }
    const char* name = PyUnicode_AsUTF8(args[0]);
    if (!name) return nullptr;
    void* address = PyLong_AsVoidPtr(args[1]);
    if (PyErr_Occurred()) return nullptr;
    for (int i = 0; i < LAUNCHERS; ++i)
        if (std::strcmp(name, LAUNCHER_NAMES[i]) == 0) { g_launcher[i] = address; return none(); }
    PyErr_Format(PyExc_ValueError, "no launcher %s", name);
    return nullptr;
}
// a device that ppml_hip_init has seen, once every launcher is bound
PyObject* ready(PyObject*, PyObject* device) {
    const long i = PyLong_AsLong(device);
    if (i == -1 && PyErr_Occurred()) return nullptr;
    for (void* p : g_launcher) if (!p) return none();
    if (i >= 0 && i < 64) g_ready.fetch_or(1ull << i, std::memory_order_release);
    return none();
}
PyObject* forget(PyObject*, PyObject*) {
    g_ready.store(0);
    return none();
}

#define FAST(f_) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f_)), METH_FASTCALL
PyMethodDef methods[] = {
    {"mul_mat", FAST(linear<MUL_MAT>), nullptr},
    {"mul_mat_f16", FAST(linear<MUL_MAT_F16>), nullptr},
    {"mul_mat_q8", FAST(mul_mat_q8), nullptr},
    {"outer_product_mean", FAST(outer_product_mean), nullptr},
    {"outer_prod_mean_back", FAST(outer_prod_mean_back), nullptr},
    {"tri_mul", FAST(tri_mul), nullptr},
    {"tri_mul_back", FAST(tri_mul_back), nullptr},
    {"flash_attn_forward", FAST(flash_attn_forward), nullptr},
    {"flash_attn_backward", FAST(flash_attn_backward), nullptr},
    {"bind", FAST(bind), nullptr},
    {"ready", ready, METH_O, nullptr},
    {"forget", forget, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// whose class layouts this was compiled against: read before the module is imported
#define TEXT_OF_(x_) #x_
#define TEXT_OF(x_) TEXT_OF_(x_)
extern "C" __attribute__((visibility("default"))) const char host_calls_built_for[] = TEXT_OF(BUILT_FOR);

PyMODINIT_FUNC PyInit__host_calls() { return PyModule_Create(&module); }
