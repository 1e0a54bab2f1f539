// Native half of the Python binding: the calls of a model's step, whose GPU time is
// of the order of the interpreter's at decode sizes, go from torch tensors to the C ABI
// here, without ctypes structures in between. Every check of the
// arguments' values stays in the library; this file only describes tensors
// (dg_tensor) and passes the status back.
//
// Host time of a call, through ctypes -> here (us): 64 x 2112 x 7168 with its workspace
// (two launches) 22.7 -> 9.6, 1 x 256 x 512 16.0 -> 4.9, the cast of 8 x 512 with its
// two allocations 15.1 -> 7.9.
//
// The entry points' addresses come from the ctypes-loaded library (init), so both
// bindings use the same one, whichever that is.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <stdexcept>
#include <string>

#include "deepgemm_mi355x.h"

namespace {

struct EntryPoints {
    decltype(&dg_fp8_fp4_gemm_nt) gemm_nt;
    decltype(&dg_fp8_fp4_gemm_nt_ws) gemm_nt_ws;
    decltype(&dg_fp8_gemm_nt_workspace_size) workspace_size;
    decltype(&dg_m_grouped_fp8_fp4_gemm_nt_contiguous) contiguous;
    decltype(&dg_m_grouped_fp8_fp4_gemm_nt_masked) masked;
    decltype(&dg_per_token_cast_to_fp8) cast;
    decltype(&dg_moe_dispatch) dispatch;
    decltype(&dg_moe_swiglu_apply_weight_to_fp8) swiglu;
    decltype(&dg_m_grouped_fp8_gemm_nt_contiguous_swiglu) contiguous_swiglu;
    decltype(&dg_m_grouped_fp8_gemm_nt_masked_swiglu) masked_swiglu;
    decltype(&dg_moe_combine) combine;
} g_entry{};

struct TypeMismatch : std::runtime_error {
    using std::runtime_error::runtime_error;
};

// DG_* code of a tensor's type, or -1 (as the ctypes binding's table).
int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return DG_F32;
        case at::kBFloat16: return DG_BF16;
        case at::kFloat8_e4m3fn: return DG_E4M3;
        case at::kInt: return DG_I32;
        case at::kChar: return DG_I8;
        case at::kByte: return DG_U8;
        case at::kHalf: return DG_F16;
        case at::kLong: return DG_I64;
        case at::ScalarType::Float4_e2m1fn_x2: return DG_I8;
        default: return -1;
    }
}

const at::Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) throw TypeMismatch(std::string("expected a torch.Tensor, got ") + Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}

// A described argument: the struct, and NULL for None where the ABI takes NULL.
struct Arg {
    dg_tensor d{};
    bool given = true;

    void fill(const at::Tensor& t) {
        const int code = dtype_code(t.scalar_type());
        if (code < 0)
            throw std::runtime_error(std::string("Assertion error (_ffi.py): unsupported dtype ") +
                                     c10::toString(t.scalar_type()));
        const auto sizes = t.sizes();
        const auto strides = t.strides();
        if (sizes.size() > 4)
            throw std::runtime_error("Assertion error (_ffi.py): tensors of rank > 4 are not supported");
        d.data = t.data_ptr();
        d.dtype = code;
        d.ndim = (int32_t)sizes.size();
        for (size_t i = 0; i < sizes.size(); ++i) {
            d.sizes[i] = sizes[i];
            d.strides[i] = strides[i];
        }
        d.device = t.is_cuda() ? (int32_t)t.get_device() : -1;
    }
    Arg() : given(false) {}
    explicit Arg(PyObject* o, bool optional = false) {
        if (optional && o == Py_None) given = false;
        else fill(tensor(o));
    }
    const dg_tensor* get() const { return given ? &d : nullptr; }
};

// Integers; a pointer argument (a ctypes structure's address) is 0 for NULL.
int64_t integer(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw TypeMismatch("");
    return v;
}
float real(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw TypeMismatch("");
    return (float)v;
}
template <typename T>
T* pointer(PyObject* o) {
    void* p = PyLong_AsVoidPtr(o);
    if (p == nullptr && PyErr_Occurred()) throw TypeMismatch("");
    return static_cast<T*>(p);
}

// Runs f without the GIL: a launch blocks while the stream's queue is full (or its module
// loads), an allocation while the device synchronizes, and the other threads run
// meanwhile, as through ctypes. f sees plain values and C++ tensors only.
template <typename F>
auto unlocked(F&& f) {
    struct Released {
        PyThreadState* state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
    } released;
    return f();
}
template <typename E, typename... A>
int32_t call(E entry, A... args) {
    return unlocked([&] { return entry(args...); });
}

// Runs f with exceptions turned into Python's: nothing leaves these functions.
template <typename F>
PyObject* guarded(Py_ssize_t nargs, Py_ssize_t want, F&& f) {
    if (nargs != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, nargs);
        return nullptr;
    }
    try {
        return PyLong_FromLong(f());
    } catch (const TypeMismatch& e) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, e.what());
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
    }
    return nullptr;
}

// init(addresses of the entry points, in EntryPoints' order)
PyObject* init(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 11, [&] {
        auto set = [&](auto& entry, int i) { entry = reinterpret_cast<std::decay_t<decltype(entry)>>(pointer<void>(a[i])); };
        set(g_entry.gemm_nt, 0), set(g_entry.gemm_nt_ws, 1), set(g_entry.workspace_size, 2);
        set(g_entry.contiguous, 3), set(g_entry.masked, 4), set(g_entry.cast, 5), set(g_entry.dispatch, 6);
        set(g_entry.swiglu, 7), set(g_entry.contiguous_swiglu, 8), set(g_entry.masked_swiglu, 9);
        set(g_entry.combine, 10);
        return 0;
    });
}

// gemm_nt(a, sfa, b, sfb, d, c | None, recipe, disable_ue8m0_cast, epilogue, stream)
PyObject* gemm_nt(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 10, [&] {
        const Arg ta(a[0]), sfa(a[1]), tb(a[2]), sfb(a[3]), d(a[4]), c(a[5], true);
        const auto* recipe = pointer<const dg_recipe>(a[6]);
        const auto disable = (int32_t)integer(a[7]);
        const auto* epilogue = pointer<const dg_epilogue>(a[8]);
        void* stream = pointer<void>(a[9]);
        // Decode-sized calls (at most 64 rows) split K over workgroups when given a
        // workspace: it comes from torch's caching allocator on the output's device
        // and current stream, and goes back to it once the launches are queued.
        if (!c.given && ta.d.ndim == 2 && tb.d.ndim > 0 && ta.d.sizes[0] <= 64 && d.d.dtype == DG_BF16) {
            const int64_t bytes = g_entry.workspace_size(ta.d.sizes[0], tb.d.sizes[0], ta.d.sizes[1]);
            if (bytes > 0) {
                const auto options = tensor(a[4]).options().dtype(at::kByte);
                const at::Tensor ws = unlocked([&] { return at::empty({bytes}, options); });
                Arg w;
                w.fill(ws);
                return call(g_entry.gemm_nt_ws, ta.get(), sfa.get(), tb.get(), sfb.get(), d.get(), nullptr, recipe,
                            disable, epilogue, &w.d, stream);
            }
        }
        return call(g_entry.gemm_nt, ta.get(), sfa.get(), tb.get(), sfb.get(), d.get(), c.get(), recipe, disable,
                    epilogue, stream);
    });
}

// contiguous(a, sfa, b, sfb, d, layout, recipe, disable, psum, zero_padding, expected_m, epilogue, stream)
PyObject* contiguous(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 13, [&] {
        const Arg ta(a[0]), sfa(a[1]), tb(a[2]), sfb(a[3]), d(a[4]), layout(a[5]);
        return call(g_entry.contiguous, ta.get(), sfa.get(), tb.get(), sfb.get(), d.get(), layout.get(),
                    pointer<const dg_recipe>(a[6]), (int32_t)integer(a[7]), (int32_t)integer(a[8]),
                    (int32_t)integer(a[9]), (int32_t)integer(a[10]), pointer<const dg_epilogue>(a[11]),
                    pointer<void>(a[12]));
    });
}

// masked(a, sfa, b, sfb, d, masked_m, expected_m, recipe, disable, epilogue, stream)
PyObject* masked(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 11, [&] {
        const Arg ta(a[0]), sfa(a[1]), tb(a[2]), sfb(a[3]), d(a[4]), masked_m(a[5]);
        return call(g_entry.masked, ta.get(), sfa.get(), tb.get(), sfb.get(), d.get(), masked_m.get(),
                    (int32_t)integer(a[6]), pointer<const dg_recipe>(a[7]), (int32_t)integer(a[8]),
                    pointer<const dg_epilogue>(a[9]), pointer<void>(a[10]));
    });
}

// cast(x, q, sf, gran_k, use_ue8m0, stream)
PyObject* cast(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 6, [&] {
        const Arg x(a[0]), q(a[1]), sf(a[2]);
        return call(g_entry.cast, x.get(), q.get(), sf.get(), (int32_t)integer(a[3]), (int32_t)integer(a[4]),
                    pointer<void>(a[5]));
    });
}

// dispatch(x, x_sf, topk, topk_weights | None, experts, layout, alignment, a, sf, grouped_layout, pos,
//          row_weights | None, workspace, stream)
PyObject* dispatch(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 14, [&] {
        const Arg x(a[0]), x_sf(a[1]), topk(a[2]), topk_w(a[3], true), out(a[7]), sf(a[8]), layout(a[9]), pos(a[10]),
            w(a[11], true), ws(a[12]);
        return call(g_entry.dispatch, x.get(), x_sf.get(), topk.get(), topk_w.get(), (int32_t)integer(a[4]),
                    (int32_t)integer(a[5]), (int32_t)integer(a[6]), out.get(), sf.get(), layout.get(), pos.get(),
                    w.get(), ws.get(), pointer<void>(a[13]));
    });
}

// swiglu(x, row_weights | None, row_layout | None, clamp, q, sf, gran_k, stream)
PyObject* swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 8, [&] {
        const Arg x(a[0]), w(a[1], true), layout(a[2], true), q(a[4]), sf(a[5]);
        return call(g_entry.swiglu, x.get(), w.get(), layout.get(), real(a[3]), q.get(), sf.get(),
                    (int32_t)integer(a[6]), pointer<void>(a[7]));
    });
}

// contiguous_swiglu(a, sfa, b, sfb, layout, row_weights | None, clamp, q, sf, psum, zero_padding, stream)
PyObject* contiguous_swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 12, [&] {
        const Arg ta(a[0]), sfa(a[1]), tb(a[2]), sfb(a[3]), layout(a[4]), w(a[5], true), q(a[7]), sf(a[8]);
        return call(g_entry.contiguous_swiglu, ta.get(), sfa.get(), tb.get(), sfb.get(), layout.get(), w.get(),
                    real(a[6]), q.get(), sf.get(), (int32_t)integer(a[9]), (int32_t)integer(a[10]),
                    pointer<void>(a[11]));
    });
}

// masked_swiglu(a, sfa, b, sfb, masked_m, expected_m, row_weights | None, clamp, q, sf, stream)
PyObject* masked_swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 11, [&] {
        const Arg ta(a[0]), sfa(a[1]), tb(a[2]), sfb(a[3]), masked_m(a[4]), w(a[6], true), q(a[8]), sf(a[9]);
        return call(g_entry.masked_swiglu, ta.get(), sfa.get(), tb.get(), sfb.get(), masked_m.get(),
                    (int32_t)integer(a[5]), w.get(), real(a[7]), q.get(), sf.get(), pointer<void>(a[10]));
    });
}

// combine(y, pos, topk_weights | None, out, stream)
PyObject* combine(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 5, [&] {
        const Arg y(a[0]), pos(a[1]), w(a[2], true), out(a[3]);
        return call(g_entry.combine, y.get(), pos.get(), w.get(), out.get(), pointer<void>(a[4]));
    });
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}

PyMethodDef g_methods[] = {method<init>("init"),     method<gemm_nt>("gemm_nt"), method<contiguous>("contiguous"),
                           method<masked>("masked"), method<cast>("cast"),       method<dispatch>("dispatch"),
                           method<swiglu>("swiglu"), method<contiguous_swiglu>("contiguous_swiglu"),
                           method<masked_swiglu>("masked_swiglu"),               method<combine>("combine"),
                           {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_dgbind", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dgbind() { return PyModule_Create(&g_module); }
