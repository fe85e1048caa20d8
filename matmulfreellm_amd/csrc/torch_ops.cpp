// Calls on single tensors, where the host is what a user waits for: no Python between the tensor and the launch, and for the scans
// none in the backward pass either, which autograd runs on a thread of its own (a Python backward waits there for the interpreter
// lock of the thread that called it).  Measured with kernels of 4.5 and 30 us of device time behind them, per call:
//   FusedBitLinear 1 x 2048 -> 2048          19.7 us through Python and ctypes, 7.7 here (the launch alone: 3)
//   fused_recurrent_hgrn, forward + backward  172 us through Python Functions, 71 here
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mmf.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

int dtype_of(at::ScalarType t) {
    return t == at::kFloat ? MMF_F32 : t == at::kBFloat16 ? MMF_BF16 : t == at::kHalf ? MMF_F16 : -1;
}
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
// the launches go to the current device: this makes it the tensors' for the time of a call
struct OnDevice {
    int back = -1;
    explicit OnDevice(int dev) {
        const int now = c10::hip::current_device();
        if (now != dev) { back = now; c10::hip::set_device((c10::DeviceIndex)dev); }
    }
    ~OnDevice() { if (back >= 0) c10::hip::set_device((c10::DeviceIndex)back); }
};
struct Failed { int rc; const char* what; };
void check(int rc, const char* what) { if (rc != 0) throw Failed{rc, what}; }

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// ------------------------------------------------------------------------------ BitLinear
// (x, norm_weight, packed, wdeq, seg_rows, n, k, eps, most_rows) -> [..., n], or None where an operand is not laid out for the launches or
// they refuse it (the general path then says why).  Up to most_rows rows run as the one fused launch, more as quantiser + contraction
// with one allocation for what passes between them.
PyObject* bitlinear(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 9) { PyErr_SetString(PyExc_TypeError, "bitlinear takes 9 arguments"); return nullptr; }
    for (int i = 0; i < 4; ++i)
        if (!THPVariable_Check(args[i])) Py_RETURN_NONE;
    const Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]), &packed = THPVariable_Unpack(args[2]),
                 &wdeq = THPVariable_Unpack(args[3]);
    const int64_t seg_rows = PyLong_AsLongLong(args[4]), n = PyLong_AsLongLong(args[5]), k = PyLong_AsLongLong(args[6]);
    const double eps = PyFloat_AsDouble(args[7]);
    const int64_t most = PyLong_AsLongLong(args[8]);
    if (PyErr_Occurred()) return nullptr;
    const int dt = dtype_of(x.scalar_type()), wdt = dtype_of(w.scalar_type());
    const int64_t total = x.numel();
    if (dt < 0 || wdt < 0 || x.dim() < 1 || x.size(-1) != k || total == 0 || !x.is_cuda() || !x.is_contiguous() ||
        !w.is_contiguous() || w.numel() != k || w.device() != x.device() || packed.device() != x.device())
        Py_RETURN_NONE;
    Tensor out;
    int rc;
    {
        NoGil nogil;
        OnDevice on(x.get_device());
        c10::SmallVector<int64_t, 6> shape(x.sizes().begin(), x.sizes().end());
        shape.back() = n;
        out = at::empty(shape, x.options().requires_grad(false));
        const int64_t rows = total / k;
        if (rows > most || k > mmf_bitlinear_gemv_max_k()) {
            const int64_t codes = mmf_codes_bytes(rows, k, 1);          // a multiple of 16 bytes
            Tensor ws = at::empty({codes + 8 * rows}, x.options().dtype(at::kByte).requires_grad(false));
            int8_t* q = static_cast<int8_t*>(ws.data_ptr());
            float* deq = reinterpret_cast<float*>(q + codes);
            int* qsum = reinterpret_cast<int*>(deq + rows);
            rc = mmf_rmsnorm_quant(x.data_ptr(), nullptr, w.data_ptr(), q, deq, qsum, nullptr, rows, k, (float)eps, dt, dt, wdt, 1, stream_of(x));
            if (rc == 0)
                rc = mmf_bitlinear_mfma(q, deq, qsum, packed.data_ptr(), static_cast<const float*>(wdeq.data_ptr()), seg_rows, nullptr, nullptr,
                                        out.data_ptr(), n, rows, k, n, dt, -1, stream_of(x));
        } else rc = mmf_bitlinear_gemv(x.data_ptr(), w.data_ptr(), packed.data_ptr(), static_cast<const float*>(wdeq.data_ptr()), seg_rows, nullptr,
                                 nullptr, out.data_ptr(), rows, k, n, (float)eps, dt, wdt, stream_of(x));
    }
    if (rc != 0) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------ scans, differentiable
float* floats(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }

// mmfreelm/ops/hgrn/recurrent_fuse.py:136-173 (chunk 0) and chunk.py:223-284
struct ScanFn : torch::autograd::Function<ScanFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& g, const std::optional<Tensor>& h0, bool final_state, int64_t chunk) {
        OnDevice on(x.get_device());
        const int64_t b = x.size(0), h = x.size(1), t = x.size(2), d = x.size(3);
        const int dt = dtype_of(x.scalar_type());
        const Tensor xc = x.contiguous(), gc = g.contiguous(), state = h0 ? h0->reshape({b * h, d}).to(at::kFloat).contiguous() : Tensor();
        const auto f32 = x.options().dtype(at::kFloat);
        Tensor o = at::empty(xc.sizes(), xc.options()), last, ws;
        if (final_state) last = at::empty({b, h, d}, f32);
        if (chunk > 0) {
            if (const int64_t bytes = mmf_hgrn_chunk_workspace_bytes(b * h, t, d, (int)chunk)) ws = at::empty({bytes / 4}, f32);
            check(mmf_hgrn_chunk(xc.data_ptr(), gc.data_ptr(), floats(state), o.data_ptr(), floats(last), b * h, t, d, (int)chunk, dt, floats(ws),
                                 stream_of(x)), "mmf_hgrn_chunk");
        } else {
            check(mmf_hgrn_recurrent(xc.data_ptr(), gc.data_ptr(), floats(state), o.data_ptr(), floats(last), b * h, t, d, dt, stream_of(x)),
                  "mmf_hgrn_recurrent");
        }
        ctx->save_for_backward({gc, o, state});
        ctx->saved_data["log_gates"] = chunk > 0;
        ctx->set_materialize_grads(false);
        if (!final_state) return {o};
        ctx->mark_non_differentiable({last});
        return {o, last};
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        if (!grads[0].defined()) return variable_list(5);
        const auto saved = ctx->get_saved_variables();
        const Tensor &g = saved[0], &o = saved[1], &state = saved[2];
        OnDevice on(g.get_device());
        const int64_t bh = g.size(0) * g.size(1), t = g.size(2), d = g.size(3);
        const Tensor dout = grads[0].to(g.scalar_type()).contiguous();
        Tensor dx = at::empty(g.sizes(), g.options()), dg = at::empty(g.sizes(), g.options()), ws;
        if (const int64_t bytes = mmf_hgrn_recurrent_bwd_workspace_bytes(bh, t, d)) ws = at::empty({bytes / 4}, g.options().dtype(at::kFloat));
        const int rc = mmf_hgrn_recurrent_bwd_split(g.data_ptr(), o.data_ptr(), dout.data_ptr(), floats(state), dx.data_ptr(), dg.data_ptr(), bh, t, d,
                                           ctx->saved_data["log_gates"].toBool() ? 1 : 0, dtype_of(g.scalar_type()), floats(ws),
                                           stream_of(g));
        TORCH_CHECK(rc == 0, "mmf_hgrn_recurrent_bwd_split: ", rc < 0 ? "MMF error " : "HIP error ", rc);
        return {dx, dg, Tensor(), Tensor(), Tensor()};
    }
};

// (x, g, initial state or None, final_state, chunk or 0, what raises for a return code) -> (o, final state or None); the caller has
// checked the operands
PyObject* scan(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 6 || !THPVariable_Check(args[0]) || !THPVariable_Check(args[1]) || !(args[2] == Py_None || THPVariable_Check(args[2]))) {
        PyErr_SetString(PyExc_TypeError, "scan takes (x, g, initial_state, final_state, chunk, check)");
        return nullptr;
    }
    const Tensor &x = THPVariable_Unpack(args[0]), &g = THPVariable_Unpack(args[1]);
    const std::optional<Tensor> h0 = args[2] == Py_None ? std::nullopt : std::optional<Tensor>(THPVariable_Unpack(args[2]));
    const bool final_state = PyObject_IsTrue(args[3]) == 1;
    const int64_t chunk = PyLong_AsLongLong(args[4]);
    if (PyErr_Occurred()) return nullptr;
    variable_list out;
    try {
        NoGil nogil;
        out = ScanFn::apply(x, g, h0, final_state, chunk);
    } catch (const Failed& f) {
        Py_XDECREF(PyObject_CallFunction(args[5], "is", f.rc, f.what));
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, f.what);
        return nullptr;
    }
    PyObject* o = THPVariable_Wrap(out[0]);
    PyObject* last = Py_None;
    if (out.size() > 1) last = THPVariable_Wrap(out[1]);
    else Py_INCREF(last);
    PyObject* r = PyTuple_Pack(2, o, last);
    Py_DECREF(o);
    Py_DECREF(last);
    return r;
    END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------ what a native block call takes for granted
// Whether all of this still holds for a block -- asked for every block of every forward, ~130 look-ups in 1.6 us:
// (block, (class, modules dict, parameters dict, [(module, class, dict)], [(dict, key, object)], [(dict, key)], [(dict, key, value)],
// [(class, forward, __call__)])):
//   the block is of that class and holds those two dicts; the modules below it are of theirs;
//   none of them has hooks or a forward of its own;
//   the dicts hold those objects, nothing or None, and equal values; the classes' forward and __call__ are the ones they were.
PyObject *kHooks[4], *kForward, *kCall, *kModules, *kParameters;
// 1 / 0, or -1 with an error set
int untouched(PyObject* d) {
    for (PyObject* name : kHooks) {
        PyObject* hooks = PyDict_GetItemWithError(d, name);
        if (!hooks) {
            if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, name);
            return -1;
        }
        const int any = PyObject_IsTrue(hooks);
        if (any != 0) return any < 0 ? -1 : 0;
    }
    const int own = PyDict_Contains(d, kForward);
    return own < 0 ? -1 : !own;
}
int holds(PyObject* d, PyObject* key, PyObject* object) {
    PyObject* held = PyDict_GetItemWithError(d, key);
    return !held && PyErr_Occurred() ? -1 : held == object;
}
// (the type's method cache: a tenth of what a general attribute look-up of a class costs)
bool method_is(PyObject* cls, PyObject* name, PyObject* function) {
    return _PyType_Lookup(reinterpret_cast<PyTypeObject*>(cls), name) == function;
}
int structure(PyObject* block, PyObject* facts) {
    auto fact = [&](int i) { return PyTuple_GET_ITEM(facts, i); };
    if (reinterpret_cast<PyObject*>(Py_TYPE(block)) != fact(0)) return 0;
    PyObject* d = PyObject_GenericGetDict(block, nullptr);
    if (!d) return -1;
    int ok = untouched(d);
    if (ok == 1) ok = holds(d, kModules, fact(1));
    if (ok == 1) ok = holds(d, kParameters, fact(2));
    Py_DECREF(d);
    if (ok != 1) return ok;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(fact(3)); ++i) {
        PyObject* t = PyList_GET_ITEM(fact(3), i);
        if (reinterpret_cast<PyObject*>(Py_TYPE(PyTuple_GET_ITEM(t, 0))) != PyTuple_GET_ITEM(t, 1)) return 0;
        if ((ok = untouched(PyTuple_GET_ITEM(t, 2))) != 1) return ok;
    }
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(fact(4)); ++i) {
        PyObject* t = PyList_GET_ITEM(fact(4), i);
        if ((ok = holds(PyTuple_GET_ITEM(t, 0), PyTuple_GET_ITEM(t, 1), PyTuple_GET_ITEM(t, 2))) != 1) return ok;
    }
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(fact(5)); ++i) {
        PyObject* t = PyList_GET_ITEM(fact(5), i);
        PyObject* held = PyDict_GetItemWithError(PyTuple_GET_ITEM(t, 0), PyTuple_GET_ITEM(t, 1));
        if (!held && PyErr_Occurred()) return -1;
        if (held && held != Py_None) return 0;
    }
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(fact(6)); ++i) {
        PyObject* t = PyList_GET_ITEM(fact(6), i);
        PyObject* held = PyDict_GetItemWithError(PyTuple_GET_ITEM(t, 0), PyTuple_GET_ITEM(t, 1));
        if (!held) return PyErr_Occurred() ? -1 : 0;
        if (held == PyTuple_GET_ITEM(t, 2)) continue;
        Py_INCREF(held);                                            // (an __eq__ may be anybody's)
        ok = PyObject_RichCompareBool(held, PyTuple_GET_ITEM(t, 2), Py_EQ);
        Py_DECREF(held);
        if (ok != 1) return ok;
    }
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(fact(7)); ++i) {
        PyObject* t = PyList_GET_ITEM(fact(7), i);
        if (!method_is(PyTuple_GET_ITEM(t, 0), kForward, PyTuple_GET_ITEM(t, 1)) || !method_is(PyTuple_GET_ITEM(t, 0), kCall, PyTuple_GET_ITEM(t, 2)))
            return 0;
    }
    return 1;
}
PyObject* structure_holds(PyObject*, PyObject* const* args, Py_ssize_t count) {
    bool fits = count == 2 && PyTuple_Check(args[1]) && PyTuple_GET_SIZE(args[1]) == 8;
    for (int i = 3; fits && i < 8; ++i) fits = PyList_Check(PyTuple_GET_ITEM(args[1], i));
    if (!fits) {
        PyErr_SetString(PyExc_TypeError, "structure_holds takes (block, (class, modules, parameters, 5 lists))");
        return nullptr;
    }
    const int ok = structure(args[0], args[1]);
    return ok < 0 ? nullptr : PyBool_FromLong(ok);
}

// [(dict, key, parameter, version, address)] -> whether the dicts hold those parameters, unwritten since
PyObject* parameters_hold(PyObject*, PyObject* list) {
    HANDLE_TH_ERRORS
    if (!PyList_Check(list)) { PyErr_SetString(PyExc_TypeError, "parameters_hold takes a list"); return nullptr; }
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
        PyObject* t = PyList_GET_ITEM(list, i);
        PyObject* held = PyDict_GetItemWithError(PyTuple_GET_ITEM(t, 0), PyTuple_GET_ITEM(t, 1));
        if (!held && PyErr_Occurred()) return nullptr;
        if (held != PyTuple_GET_ITEM(t, 2) || !THPVariable_Check(held)) Py_RETURN_FALSE;
        const Tensor& p = THPVariable_Unpack(held);
        if (p._version() != PyLong_AsLongLong(PyTuple_GET_ITEM(t, 3)) ||
            reinterpret_cast<uintptr_t>(p.is_meta() ? nullptr : p.data_ptr()) != (uintptr_t)PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(t, 4)))
            Py_RETURN_FALSE;
        if (PyErr_Occurred()) return nullptr;
    }
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"structure_holds", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(structure_holds)), METH_FASTCALL, nullptr},
    {"parameters_hold", parameters_hold, METH_O, nullptr},
    {"bitlinear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(bitlinear)), METH_FASTCALL, nullptr},
    {"scan", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(scan)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "mmf_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_mmf_torch() {
    const char* names[4] = {"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"};
    for (int i = 0; i < 4; ++i)
        if (!(kHooks[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
    if (!(kForward = PyUnicode_InternFromString("forward")) || !(kCall = PyUnicode_InternFromString("__call__")) ||
        !(kModules = PyUnicode_InternFromString("_modules")) || !(kParameters = PyUnicode_InternFromString("_parameters")))
        return nullptr;
    return PyModule_Create(&module);
}
