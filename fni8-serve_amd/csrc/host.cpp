// Native host path of the tensor-level entry points (module fni8serve_amd._host).
//
// A decode call is a few microseconds of GPU work, while the Python of one ops.py
// entry point (argument checks, four allocations, the ctypes call) takes about 15:
// a small eager call is bound by its host code.  These functions do the same checks,
// allocate the outputs and one scratch buffer per call, and make the C ABI calls of
// a whole chain (linear, norm, MLP, MoE) from one Python call.
//
// Every function returns None, having written nothing, unless each argument is a plain
// dense GPU tensor of the type and layout that the chain takes as it is; ops.py then
// goes the general way, which converts, copies or refuses.  The one product that goes
// through torch's dispatcher (the router's logits) is checked like an argument: a mode
// such as autocast may have changed its type.  Nothing is kept between calls.  Tensors
// come from the caching allocator on the current stream, like those of the general
// way, so the calls can be captured in a graph.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include "../../include/fni8amd.h"

namespace {

using at::Tensor;

struct Refused {};  // the general way takes this call

void need(bool ok) {
    if (!ok) throw Refused{};
}

// The tensor of an argument: a plain Tensor or Parameter backed by storage, no
// subclass and no functorch or functionalization wrapper.
const Tensor& plain(PyObject* o) {
    need(THPVariable_CheckExact(o));
    const Tensor& t = THPVariable_Unpack(o);
    constexpr auto wrapped = c10::DispatchKeySet(
        {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
         c10::DispatchKey::Sparse, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
    need(t.defined() && t.is_cuda() && !t.key_set().has_any(wrapped) && t.has_storage() &&
         t.layout() == at::kStrided);
    return t;
}

Tensor maybe(PyObject* o) { return o == Py_None ? Tensor() : plain(o); }

int64_t integer(PyObject* o) {
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}

double real(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
}

void same(const Tensor& t, const Tensor& x, at::ScalarType type) {
    need(t.scalar_type() == type && t.device() == x.device() && t.is_contiguous());
}

struct Failed {
    const char* name;
    int rc;
};

void check(const char* name, int rc) {
    if (rc != FNI8_OK) throw Failed{name, rc};
}

int64_t up256(int64_t n) { return (n + 255) & ~(int64_t)255; }

// Rows of x[..., K] as they lie: contiguous, or a 2-D view with its own row stride.
struct Rows {
    const void* p;
    int64_t M, K, ld;
};
Rows rows(const Tensor& x, at::ScalarType type) {
    need(x.scalar_type() == type && x.dim() >= 1 && x.numel() > 0);
    const int64_t K = x.size(-1), M = x.numel() / K;
    if (x.is_contiguous()) return {x.data_ptr(), M, K, K};
    need(x.dim() == 2 && x.stride(1) == 1 && (M == 1 || x.stride(0) >= K));
    return {x.data_ptr(), M, K, M == 1 ? K : x.stride(0)};
}

Tensor shaped(const Tensor& x, int64_t last, at::ScalarType type) {
    at::DimVector s(x.sizes().begin(), x.sizes().end());
    s.back() = last;
    return at::empty(s, x.options().dtype(type));
}

// A weight of either scheme: int8 [N, K] with fp32 [N] scales (G = 0), or packed
// int4 [N, K/2] with fp32 [N, K/G].
struct Weight {
    const void* w;
    const float* s;
    const void* bias;
    int64_t N, K, G;
};
Weight weight(const Tensor& w, const Tensor& s, int64_t G, const Tensor& bias, const Tensor& x,
              int64_t K) {
    need(w.dim() == 2);
    const int64_t N = w.size(0);
    same(w, x, G ? at::kByte : at::kChar);
    same(s, x, at::kFloat);
    if (G) {
        need((G == 32 || G == 64 || G == 128 || G == 256) && K % G == 0 && K % 32 == 0);
        need(2 * w.size(1) == K && s.numel() == N * (K / G));
    } else {
        need(w.size(1) == K && s.numel() == N);
    }
    if (bias.defined()) {
        same(bias, x, at::kHalf);
        need(bias.numel() == N);
    }
    return {w.data_ptr(), static_cast<const float*>(s.data_ptr()),
            bias.defined() ? bias.data_ptr() : nullptr, N, K, G};
}

// Byte ranges of one scratch allocation.
struct Scratch {
    int64_t size = 0;
    Tensor t;
    int64_t take(int64_t bytes) {
        const int64_t at = size;
        size += up256(bytes);
        return at;
    }
    void alloc(const Tensor& x) { t = at::empty({size}, x.options().dtype(at::kByte)); }
    template <class T>
    T* at_(int64_t off) const {
        return reinterpret_cast<T*>(static_cast<int8_t*>(t.data_ptr()) + off);
    }
};

// A linear's part of the scratch: quantized rows, their scales, the workspace.
struct LinearScratch {
    int64_t xq, xs, work, nw;
    LinearScratch(Scratch& sc, int64_t M, const Weight& w) {
        xq = sc.take(M * w.K);
        xs = sc.take(4 * M);
        nw = w.G ? 0 : fni8_linear_workspace_bytes(M, w.N, w.K);
        work = sc.take(nw);
    }
};

void run_linear(const Scratch& sc, const LinearScratch& l, const void* x, int64_t ldx, int64_t M,
                const Weight& w, void* y, void* st) {
    int8_t* xq = sc.at_<int8_t>(l.xq);
    float* xs = sc.at_<float>(l.xs);
    if (w.G)
        check("fni8_linear_w4a8_f16",
              fni8_linear_w4a8_f16(x, ldx, M, w.K, static_cast<const uint8_t*>(w.w), w.s, w.N, w.G,
                                   w.bias, y, w.N, xq, xs, st));
    else
        check("fni8_linear_w8a8_f16_ws",
              fni8_linear_w8a8_f16_ws(x, ldx, M, w.K, static_cast<const int8_t*>(w.w), w.s, w.N,
                                      w.bias, y, w.N, xq, xs, nullptr,
                                      l.nw ? sc.at_<int8_t>(l.work) : nullptr, l.nw, st));
}

void run_gemm(const int8_t* xq, int64_t ldq, const float* xs, int64_t M, const Weight& w, void* y,
              int8_t* work, int64_t nw, void* st) {
    if (w.G)
        check("fni8_gemm_w4a8",
              fni8_gemm_w4a8(xq, ldq, xs, M, w.K, static_cast<const uint8_t*>(w.w), w.s, w.N, w.G,
                             w.bias, y, w.N, st));
    else
        check("fni8_gemm_w8a8_ws",
              fni8_gemm_w8a8_ws(xq, ldq, xs, M, w.K, static_cast<const int8_t*>(w.w), w.s, w.N,
                                w.bias, y, w.N, nullptr, work, nw, st));
}

void* stream_of(const Tensor& x) {
    return c10::hip::getCurrentHIPStream(x.device().index()).stream();
}

// Runs `body(args)` without the interpreter lock once it has unpacked its arguments:
// body returns a closure, the closure makes the calls.  None where it is refused.
template <class Body>
PyObject* entry(PyObject* const* a, Py_ssize_t n, Py_ssize_t want, Body body) {
    HANDLE_TH_ERRORS
    if (n != want) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    if (c10::impl::TorchDispatchModeTLS::any_modes_set()) Py_RETURN_NONE;
    try {
        auto work = body(a);
        decltype(work()) out;
        {
            pybind11::gil_scoped_release no_gil;
            out = work();
        }
        return out.wrap();
    } catch (const Refused&) {
        Py_RETURN_NONE;
    } catch (const Failed& f) {
        const bool arg = f.rc == FNI8_ERR_NULL || f.rc == FNI8_ERR_SHAPE ||
                         f.rc == FNI8_ERR_ALIGN || f.rc == FNI8_ERR_STRIDE;
        PyErr_Format(arg ? PyExc_ValueError : PyExc_RuntimeError, "%s: %s: %s", f.name,
                     fni8_strerror(f.rc), fni8_last_error());
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

struct One {
    Tensor t;
    PyObject* wrap() { return THPVariable_Wrap(t); }
};
struct Several {
    Tensor t[3];
    int n = 0;
    PyObject* wrap() {
        if (n == 1) return THPVariable_Wrap(t[0]);
        PyObject* out = PyTuple_New(n);
        if (!out) throw python_error();
        for (int i = 0; i < n; i++) {
            PyObject* o = THPVariable_Wrap(t[i]);
            if (!o) {
                Py_DECREF(out);
                throw python_error();
            }
            PyTuple_SET_ITEM(out, i, o);
        }
        return out;
    }
};

// linear(x, w, scale, G, bias)
PyObject* py_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return entry(a, n, 5, [](PyObject* const* a) {
        const Tensor &x = plain(a[0]), &w = plain(a[1]), &s = plain(a[2]);
        const int64_t G = integer(a[3]);
        Tensor bias = maybe(a[4]);
        const Rows r = rows(x, at::kHalf);
        const Weight wt = weight(w, s, G, bias, x, r.K);
        return [x, wt, r] {
            c10::DeviceGuard guard(x.device());
            Scratch sc;
            const LinearScratch l(sc, r.M, wt);
            Tensor y = shaped(x, wt.N, at::kHalf);
            sc.alloc(x);
            run_linear(sc, l, r.p, r.ld, r.M, wt, y.data_ptr(), stream_of(x));
            return One{y};
        };
    });
}

// gemm(xq, xs, w, scale, G, bias)
PyObject* py_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return entry(a, n, 6, [](PyObject* const* a) {
        const Tensor &xq = plain(a[0]), &xs = plain(a[1]), &w = plain(a[2]), &s = plain(a[3]);
        const int64_t G = integer(a[4]);
        Tensor bias = maybe(a[5]);
        need(xq.dim() == 2);
        const Rows r = rows(xq, at::kChar);
        same(xs, xq, at::kFloat);
        need(xs.numel() == r.M);
        need(!G || (r.ld % 16 == 0 && reinterpret_cast<uintptr_t>(r.p) % 16 == 0));
        const Weight wt = weight(w, s, G, bias, xq, r.K);
        const float* sp = static_cast<const float*>(xs.data_ptr());
        return [xq, wt, r, sp] {
            c10::DeviceGuard guard(xq.device());
            Tensor y = at::empty({r.M, wt.N}, xq.options().dtype(at::kHalf));
            const int64_t nw = wt.G ? 0 : fni8_linear_workspace_bytes(r.M, wt.N, wt.K);
            Scratch sc;
            sc.take(nw);
            if (nw) sc.alloc(xq);
            run_gemm(static_cast<const int8_t*>(r.p), r.ld, sp, r.M, wt, y.data_ptr(),
                     nw ? sc.at_<int8_t>(0) : nullptr, nw, stream_of(xq));
            return One{y};
        };
    });
}

// mlp(x, w1, s1, G1, b1, w2, s2, G2, b2, act, fuse_min_rows): gate_up, activation,
// down; from fuse_min_rows rows the activation also quantizes for down.
PyObject* py_mlp(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return entry(a, n, 11, [](PyObject* const* a) {
        const Tensor& x = plain(a[0]);
        const Rows r = rows(x, at::kHalf);
        const Tensor b1 = maybe(a[4]), b2 = maybe(a[8]);
        const Weight up = weight(plain(a[1]), plain(a[2]), integer(a[3]), b1, x, r.K);
        need(up.N % 2 == 0);
        const int64_t I = up.N / 2;
        const Weight down = weight(plain(a[5]), plain(a[6]), integer(a[7]), b2, x, I);
        const int act = (int)integer(a[9]);
        const bool fused = r.M >= integer(a[10]);
        need(!fused || I % 4 == 0);
        need(!fused || !down.G || I % 16 == 0);
        return [x, r, up, down, I, act, fused] {
            c10::DeviceGuard guard(x.device());
            void* st = stream_of(x);
            const int64_t M = r.M;
            Scratch sc;
            const LinearScratch l1(sc, M, up);
            const int64_t h = sc.take(2 * M * up.N);
            const LinearScratch l2(sc, M, down);
            const int64_t an = fused ? fni8_act_and_mul_quant_workspace_bytes(M, I) : 2 * M * I;
            const int64_t ab = sc.take(an);
            Tensor y = shaped(x, down.N, at::kHalf);
            sc.alloc(x);
            run_linear(sc, l1, r.p, r.ld, M, up, sc.at_<void>(h), st);
            if (fused) {
                int8_t* xq = sc.at_<int8_t>(l2.xq);
                float* xs = sc.at_<float>(l2.xs);
                check("fni8_act_and_mul_quant_f16_ws",
                      fni8_act_and_mul_quant_f16_ws(sc.at_<void>(h), up.N, M, I, act, xq, I, xs,
                                                    an ? sc.at_<void>(ab) : nullptr, an, st));
                run_gemm(xq, I, xs, M, down, y.data_ptr(),
                         l2.nw ? sc.at_<int8_t>(l2.work) : nullptr, l2.nw, st);
            } else {
                check("fni8_act_and_mul_f16", fni8_act_and_mul_f16(sc.at_<void>(h), up.N, M, I, act,
                                                                   sc.at_<void>(ab), I, st));
                run_linear(sc, l2, sc.at_<void>(ab), I, M, down, y.data_ptr(), st);
            }
            return One{y};
        };
    });
}

// rmsnorm(x, weight, eps, residual, unit_offset, quant) -> normed or (xq, xs), then
// x + residual with a residual
PyObject* py_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return entry(a, n, 6, [](PyObject* const* a) {
        const Tensor &x = plain(a[0]), &w = plain(a[1]);
        const float eps = (float)real(a[2]);
        const Tensor res = maybe(a[3]);
        const int unit = PyObject_IsTrue(a[4]), quant = PyObject_IsTrue(a[5]);
        const Rows r = rows(x, at::kHalf);
        same(w, x, at::kHalf);
        need(w.numel() == r.K && (!quant || r.K % 4 == 0));
        const void* rp = nullptr;
        if (res.defined()) {
            same(res, x, at::kHalf);
            need(res.sizes() == x.sizes());
            rp = res.data_ptr();
        }
        const void* wp = w.data_ptr();
        return [x, r, wp, rp, eps, unit, quant] {
            c10::DeviceGuard guard(x.device());
            void* st = stream_of(x);
            Several out;
            Tensor sum;
            if (rp) sum = at::empty(x.sizes(), x.options());
            void* sp = rp ? sum.data_ptr() : nullptr;
            if (quant) {
                Tensor xq = at::empty({r.M, r.K}, x.options().dtype(at::kChar));
                Tensor xs = at::empty({r.M}, x.options().dtype(at::kFloat));
                check("fni8_rmsnorm_quant_f16",
                      fni8_rmsnorm_quant_f16(r.p, r.ld, rp, rp ? r.K : 0, wp, eps, unit, r.M, r.K,
                                             static_cast<int8_t*>(xq.data_ptr()), r.K,
                                             static_cast<float*>(xs.data_ptr()), sp, r.K, st));
                out.t[out.n++] = xq;
                out.t[out.n++] = xs;
            } else {
                Tensor y = at::empty(x.sizes(), x.options());
                check("fni8_rmsnorm_f16",
                      fni8_rmsnorm_f16(r.p, r.ld, rp, rp ? r.K : 0, wp, eps, unit, r.M, r.K,
                                       y.data_ptr(), r.K, sp, r.K, st));
                out.t[out.n++] = y;
            }
            if (rp) out.t[out.n++] = sum;
            return out;
        };
    });
}

// Stacked expert weights [E, N, K] (or [E, N, K/2] packed) and scales.
Weight stacked(const Tensor& w, const Tensor& s, int64_t G, const Tensor& x, int64_t E, int64_t K) {
    need(w.dim() == 3 && w.size(0) == E);
    const int64_t N = w.size(1);
    same(w, x, G ? at::kByte : at::kChar);
    same(s, x, at::kFloat);
    if (G)
        need((G == 64 || G == 128 || G == 256) && K % 256 == 0 && 2 * w.size(2) == K &&
             s.numel() == E * N * (K / G));
    else
        need(w.size(2) == K && s.numel() == E * N);
    return {w.data_ptr(), static_cast<const float*>(s.data_ptr()), nullptr, N, K, G};
}

void run_grouped(const int8_t* xq, const float* xs, const int32_t* map, int64_t R, const Weight& w,
                 int64_t E, const int32_t* seg, void* y, void* st) {
    if (w.G)
        check("fni8_gemm_w4a8_grouped",
              fni8_gemm_w4a8_grouped(xq, xs, map, R, w.K, static_cast<const uint8_t*>(w.w), w.s, E,
                                     w.N, w.G, seg, nullptr, y, st));
    else
        check("fni8_gemm_w8a8_grouped",
              fni8_gemm_w8a8_grouped(xq, xs, map, R, w.K, static_cast<const int8_t*>(w.w), w.s, E,
                                     w.N, seg, nullptr, y, nullptr, st));
}

// moe(x, gate_f32, score_bias, scoring, groups, topk_group, k, renorm, scale,
//     w_gate_up, s_gate_up, G1, w_down, s_down, G2, act): the routed experts' output.
PyObject* py_moe(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return entry(a, n, 16, [](PyObject* const* a) {
        const Tensor &x = plain(a[0]), &gate = plain(a[1]);
        const Tensor sbias = maybe(a[2]);
        need(x.dim() == 2 && x.is_contiguous());
        const Rows r = rows(x, at::kHalf);
        need(gate.dim() == 2 && gate.size(1) == r.K);
        same(gate, x, at::kFloat);
        const int64_t E = gate.size(0), k = integer(a[6]);
        if (sbias.defined()) {
            same(sbias, x, at::kFloat);
            need(sbias.numel() == E);
        }
        const int scoring = (int)integer(a[3]), renorm = PyObject_IsTrue(a[7]);
        const int64_t groups = integer(a[4]), tgroup = integer(a[5]);
        const float scale = (float)real(a[8]);
        const Weight up = stacked(plain(a[9]), plain(a[10]), integer(a[11]), x, E, r.K);
        need(up.N % 8 == 0);
        const int64_t I = up.N / 2;
        const Weight down = stacked(plain(a[12]), plain(a[13]), integer(a[14]), x, E, I);
        need(down.N == r.K);
        const int act = (int)integer(a[15]);
        return [=, x = x, gate = gate, sbias = sbias] {
            c10::DeviceGuard guard(x.device());
            void* st = stream_of(x);
            const int64_t T = r.M, H = r.K, R = T * k;
            // a dispatched product: under autocast it comes back in 16 bits, which
            // the general way refuses
            const Tensor logits = at::linear(x.to(at::kFloat), gate);
            need(logits.scalar_type() == at::kFloat && logits.is_contiguous() &&
                 logits.dim() == 2 && logits.size(0) == T && logits.size(1) == E);
            Scratch sc;
            const int64_t topw = sc.take(2 * R), topi = sc.take(4 * R), seg = sc.take(4 * (E + 1)),
                          map = sc.take(4 * R), pos = sc.take(4 * R), xq = sc.take(T * H),
                          xs = sc.take(4 * T), h = sc.take(2 * R * up.N), aq = sc.take(R * I),
                          as = sc.take(4 * R), ys = sc.take(2 * R * H);
            const int64_t an = fni8_act_and_mul_quant_workspace_bytes(R, I), ab = sc.take(an);
            Tensor out = at::empty({T, H}, x.options());
            sc.alloc(x);
            int32_t *ti = sc.at_<int32_t>(topi), *sg = sc.at_<int32_t>(seg),
                    *mp = sc.at_<int32_t>(map), *ps = sc.at_<int32_t>(pos);
            check("fni8_moe_route",
                  fni8_moe_route(static_cast<const float*>(logits.data_ptr()), T, E, E, scoring,
                                 sbias.defined() ? static_cast<const float*>(sbias.data_ptr()) : nullptr,
                                 groups, tgroup, k, renorm, scale, sc.at_<void>(topw), ti, st));
            check("fni8_moe_sort", fni8_moe_sort(ti, T, k, E, sg, mp, ps, st));
            check("fni8_quantize_rowwise_f16",
                  fni8_quantize_rowwise_f16(r.p, T, H, H, sc.at_<int8_t>(xq), H, sc.at_<float>(xs), st));
            run_grouped(sc.at_<int8_t>(xq), sc.at_<float>(xs), mp, R, up, E, sg, sc.at_<void>(h), st);
            check("fni8_act_and_mul_quant_f16_ws",
                  fni8_act_and_mul_quant_f16_ws(sc.at_<void>(h), up.N, R, I, act, sc.at_<int8_t>(aq),
                                                I, sc.at_<float>(as),
                                                an ? sc.at_<void>(ab) : nullptr, an, st));
            run_grouped(sc.at_<int8_t>(aq), sc.at_<float>(as), nullptr, R, down, E, sg,
                        sc.at_<void>(ys), st);
            check("fni8_moe_combine_f16",
                  fni8_moe_combine_f16(sc.at_<void>(ys), H, ti, sc.at_<void>(topw), ps, T, k,
                                       out.data_ptr(), st));
            return One{out};
        };
    });
}

#define FNI8_METHOD(name) \
    {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FNI8_METHOD(linear), FNI8_METHOD(gemm), FNI8_METHOD(mlp),
                         FNI8_METHOD(rmsnorm), FNI8_METHOD(moe), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: the torch this was compiled against, which _lib.py compares before
// the first call (torch's C++ ABI holds for one build only).
PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", FNI8_TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
