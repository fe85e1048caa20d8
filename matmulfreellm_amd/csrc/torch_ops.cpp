// Calls on single tensors, where the host is what a user waits for: no Python between the tensor and the launch, and for the scans
// none in the backward pass either, which autograd runs on a thread of its own (a Python backward waits there for the interpreter
// lock of the thread that called it).  Measured with kernels of 4.5 and 30 us of device time behind them, per call:
//   FusedBitLinear 1 x 2048 -> 2048          19.7 us through Python and ctypes, 7.7 here (the launch alone: 3)
//   fused_recurrent_hgrn, forward + backward  172 us through Python Functions, 71 here
//   the backward of a block, ~30 launches      359 us through Python and ctypes, 239 here
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
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
// null, with the exception that `raise`, a caller's function of (code, name), makes of a failure
PyObject* failed(const Failed& f, PyObject* raise) {
    Py_XDECREF(PyObject_CallFunction(raise, "is", f.rc, f.what));
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, f.what);
    return nullptr;
}
// None is an undefined tensor
bool tensor_or_none(PyObject* o, Tensor& t) {
    if (THPVariable_Check(o)) t = THPVariable_Unpack(o);
    return THPVariable_Check(o) || o == Py_None;
}

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
        return failed(f, args[5]);
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

// ------------------------------------------------------------------------------ backward of a block
enum Chain : int { CHAIN_NORM = 0, CHAIN_GATED = 1, CHAIN_SWIGLU = 2, CHAIN_RESNORM = 3 };
void* address(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

struct Chained { Tensor dx, y, dw; };
// mmf_chain_bwd over [M, K] operands (column slices keep their row stride; dy: one [M, K] a norm); dx is allocated unless given
Chained chain(int kind, const Tensor& x, const Tensor& aux, const Tensor& w1, double eps1, at::ArrayRef<Tensor> w2, double eps2, at::ArrayRef<Tensor> dy,
              const Tensor& dres, Tensor dx, const Tensor& daux) {
    const int64_t m = x.size(0), k = x.size(1), n = (int64_t)w2.size(), rows = n + (kind != CHAIN_SWIGLU);
    if (!dx.defined()) dx = at::empty({m, k}, x.options());
    Tensor y = at::empty({n, m, k}, x.options()), dw = at::empty({rows, k}, w2[0].options());
    Tensor part = at::empty({mmf_chain_bwd_groups(m) * rows * k}, x.options().dtype(at::kFloat));
    const void *w2p[3] = {}, *dyp[3] = {};
    for (int64_t i = 0; i < n; ++i) {
        w2p[i] = w2[i].data_ptr();
        dyp[i] = dy[i].data_ptr();
    }
    check(mmf_chain_bwd(kind, x.data_ptr(), x.stride(0), address(aux), aux.defined() ? aux.stride(0) : 0, address(w1), (float)eps1, (int)n, w2p,
                        (float)eps2, dyp, k, address(dres), dx.data_ptr(), dx.stride(0), address(daux), daux.defined() ? daux.stride(0) : 0, y.data_ptr(),
                        floats(part), dw.data_ptr(), m, k, dtype_of(x.scalar_type()), dtype_of(dw.scalar_type()), stream_of(x)),
          "mmf_chain_bwd");
    return {dx, y, dw};
}

struct Packed { Tensor codes, wdeq; int64_t seg_rows, n, k; };
// t * wdeq as a dense [N, K] matrix for dout @ W_q (fusedbitnet.py:456-458), stored as that product and its unpacking take least time together.  16-bit
// products run faster with the contraction, N, contiguous.  Single-precision ones take the same time either way, and rows are written faster than
// columns: a 1024-wide step's 13 unpackings 126 us stored [K, N], 103 us stored [N, K].
Tensor dense(const Packed& p, const at::TensorOptions& like) {
    const auto type = c10::typeMetaToScalarType(like.dtype());
    const bool rows = type == at::kFloat;
    Tensor w = rows ? at::empty({p.n, p.k}, like) : at::empty({p.k, p.n}, like);
    check((rows ? mmf_unpack_dequant : mmf_unpack_dequant_t)(p.codes.data_ptr(), floats(p.wdeq), p.seg_rows, p.n, p.k, w.data_ptr(), dtype_of(type),
                                                             stream_of(w)),
          rows ? "mmf_unpack_dequant" : "mmf_unpack_dequant_t");
    return rows ? w : w.t();
}

// (kind, x, aux or None, w1 or None, eps1, norm weights, eps2, their gradients, dres or None, dx or None, daux or None, what raises for a return code) ->
// (dx, y [norms, M, K], weight gradients [(w1) + norms, K]); daux is written where it is given
PyObject* chain_backward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    Tensor x, aux, w1, dres, dx, daux, w2[3], dy[3];
    bool fits = count == 12 && THPVariable_Check(args[1]) && tensor_or_none(args[1], x) && tensor_or_none(args[2], aux) && tensor_or_none(args[3], w1) &&
                PyTuple_Check(args[5]) && PyTuple_Check(args[7]) && tensor_or_none(args[8], dres) && tensor_or_none(args[9], dx) && tensor_or_none(args[10], daux);
    const Py_ssize_t n = fits ? PyTuple_GET_SIZE(args[5]) : 0;
    fits = fits && n >= 1 && n <= 3 && PyTuple_GET_SIZE(args[7]) == n && x.dim() == 2;
    for (Py_ssize_t i = 0; fits && i < n; ++i) {
        PyObject *w = PyTuple_GET_ITEM(args[5], i), *d = PyTuple_GET_ITEM(args[7], i);
        fits = THPVariable_Check(w) && THPVariable_Check(d) && tensor_or_none(w, w2[i]) && tensor_or_none(d, dy[i]);
    }
    if (!fits) {
        PyErr_SetString(PyExc_TypeError, "chain_backward takes (kind, x, aux, w1, eps1, w2, eps2, dy, dres, dx, daux, check)");
        return nullptr;
    }
    const int kind = (int)PyLong_AsLong(args[0]);
    const double eps1 = PyFloat_AsDouble(args[4]), eps2 = PyFloat_AsDouble(args[6]);
    if (PyErr_Occurred()) return nullptr;
    Chained c;
    try {
        NoGil nogil;
        OnDevice on(x.get_device());
        c = chain(kind, x, aux, w1, eps1, at::ArrayRef<Tensor>(w2, n), eps2, at::ArrayRef<Tensor>(dy, n), dres, dx, daux);
    } catch (const Failed& f) {
        return failed(f, args[11]);
    }
    PyObject *a = THPVariable_Wrap(c.dx), *b = THPVariable_Wrap(c.y), *w = THPVariable_Wrap(c.dw), *r = PyTuple_Pack(3, a, b, w);
    Py_DECREF(a);
    Py_DECREF(b);
    Py_DECREF(w);
    return r;
    END_HANDLE_TH_ERRORS
}

// (codes, wdeq, seg_rows, n, k, dtype, what raises for a return code) -> [n, k]
PyObject* dense_weight(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 7 || !THPVariable_Check(args[0]) || !THPVariable_Check(args[1]) || !THPDtype_Check(args[5])) {
        PyErr_SetString(PyExc_TypeError, "dense_weight takes (codes, wdeq, seg_rows, n, k, dtype, check)");
        return nullptr;
    }
    const Packed p{THPVariable_Unpack(args[0]), THPVariable_Unpack(args[1]), PyLong_AsLongLong(args[2]), PyLong_AsLongLong(args[3]), PyLong_AsLongLong(args[4])};
    if (PyErr_Occurred()) return nullptr;
    const auto type = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
    Tensor w;
    try {
        NoGil nogil;
        OnDevice on(p.codes.get_device());
        w = dense(p, p.codes.options().dtype(type));
    } catch (const Failed& f) {
        return failed(f, args[6]);
    }
    return THPVariable_Wrap(std::move(w));
    END_HANDLE_TH_ERRORS
}

// dout^T @ y of a block's BitLinears, [M, N] gradients and [M, K] de-quantised inputs; undefined where a gradient is.
// Two or more go in one launch: each by itself leaves much of the chip idle, or its launch takes longer than it does.  The six of a
// block, one library product each / together, us: bf16, 2048 wide 64 rows 114 / 41, 1024 186 / 123, 8192 916 / 716; 1024 wide 112 / 34
// and 456 / 206 (1024, 8192 rows); fp32, 1024 wide 666 rows 220 / 143, 2048 wide 591 / 514 and 1522 / 1487 (666, 2002 rows).  One alone
// (2048 x 2048, bf16: 1024 rows 21 / 29, 8192 86 / 81) stays with the library, and so do many rows of wide blocks in fp32, where each
// product fills the chip (2048 wide, 4096 rows 2859 / 2999; 1536 wide 1659 / 1671; 1024 wide 801 / 783).
std::vector<Tensor> weight_grads(at::ArrayRef<std::pair<Tensor, Tensor>> pairs) {
    std::vector<Tensor> out(pairs.size());
    const void *p[8], *q[8];
    void* o[8];
    int64_t ldp[8], ldq[8], n[8], k[8], outputs = 0;
    int count = 0, which[8];
    for (size_t i = 0; i < pairs.size(); ++i) {
        const Tensor &d = pairs[i].first, &y = pairs[i].second;
        if (!d.defined() || dtype_of(y.scalar_type()) < 0 || d.scalar_type() != y.scalar_type() || d.size(0) < 1 || d.size(0) > 0x7fffffff) continue;
        const int64_t whole = 16 / (int64_t)y.element_size();
        auto turns = [&](const Tensor& t) {
            return t.stride(1) == 1 && t.size(1) > 0 && t.size(1) % whole == 0 && t.stride(0) % whole == 0 && t.size(1) <= t.stride(0) &&
                   t.stride(0) <= 1 << 24 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
        };
        if (!turns(d) || !turns(y)) continue;
        p[count] = d.data_ptr();
        q[count] = y.data_ptr();
        ldp[count] = d.stride(0);
        ldq[count] = y.stride(0);
        n[count] = d.size(1);
        k[count] = y.size(1);
        outputs += d.size(1) * y.size(1);
        which[count++] = (int)i;
    }
    if (count >= 2) {
        const Tensor& y = pairs[which[0]].second;
        const int64_t m = y.size(0);
        const int dt = dtype_of(y.scalar_type());
        if (dt != MMF_F32 || m <= 2048 || outputs <= 1 << 24) {
            for (int i = 0; i < count; ++i) o[i] = (out[which[i]] = at::empty({n[i], k[i]}, y.options())).data_ptr();
            Tensor ws;
            if (const int64_t bytes = mmf_weight_grad_workspace_bytes(count, n, k, m, dt)) ws = at::empty({bytes}, y.options().dtype(at::kByte));
            check(mmf_weight_grad(count, p, ldp, q, ldq, o, n, k, m, dt, address(ws), stream_of(y)), "mmf_weight_grad");
        }
    }
    for (size_t i = 0; i < pairs.size(); ++i)
        if (!out[i].defined() && pairs[i].first.defined()) out[i] = at::mm(pairs[i].first.t(), pairs[i].second);
    return out;
}

// (dout [M, H], (B, T), (H, D, I), (x, lower_bound or None, mask or None, ifg, xg, o, attn, y, the nine norm weights), 4 packed weights (codes,
// wdeq, seg_rows, n, k) of the stacked projection, o, gate, down, 7 eps (attn, ifg, g, o, mlp, gate, down), the six weights' needs, what raises
// for a return code) -> (dx, d lower_bound, dw of ifg's / o's / gate's / down's chains, the six weight gradients)
PyObject* block_backward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    bool fits = count == 8 && THPVariable_Check(args[0]);
    for (int i = 1; fits && i < 7; ++i) fits = PyTuple_Check(args[i]);
    if (fits) fits = PyTuple_GET_SIZE(args[1]) == 2 && PyTuple_GET_SIZE(args[2]) == 3 && PyTuple_GET_SIZE(args[3]) == 17 && PyTuple_GET_SIZE(args[4]) == 4 &&
                     PyTuple_GET_SIZE(args[5]) == 7 && PyTuple_GET_SIZE(args[6]) == 6;
    Tensor s[17];
    for (int i = 0; fits && i < 17; ++i) {
        PyObject* t = PyTuple_GET_ITEM(args[3], i);
        if (THPVariable_Check(t)) s[i] = THPVariable_Unpack(t);
        else fits = t == Py_None && (i == 1 || i == 2);
    }
    Packed pw[4];
    for (int i = 0; fits && i < 4; ++i) {
        PyObject* t = PyTuple_GET_ITEM(args[4], i);
        if (!(fits = PyTuple_Check(t) && PyTuple_GET_SIZE(t) == 5 && THPVariable_Check(PyTuple_GET_ITEM(t, 0)) && THPVariable_Check(PyTuple_GET_ITEM(t, 1)))) break;
        pw[i] = Packed{THPVariable_Unpack(PyTuple_GET_ITEM(t, 0)), THPVariable_Unpack(PyTuple_GET_ITEM(t, 1)), PyLong_AsLongLong(PyTuple_GET_ITEM(t, 2)),
                       PyLong_AsLongLong(PyTuple_GET_ITEM(t, 3)), PyLong_AsLongLong(PyTuple_GET_ITEM(t, 4))};
    }
    if (!fits) {
        PyErr_SetString(PyExc_TypeError, "block_backward takes (dout, (B, T), (H, D, I), 17 saved, 4 packed weights, 7 eps, 6 needs, check)");
        return nullptr;
    }
    auto whole = [&](int a, int i) { return (int64_t)PyLong_AsLongLong(PyTuple_GET_ITEM(args[a], i)); };
    const int64_t b = whole(1, 0), t = whole(1, 1), H = whole(2, 0), D = whole(2, 1), I = whole(2, 2), m = b * t;
    double eps[7];
    int need[6];
    for (int i = 0; i < 7; ++i) eps[i] = PyFloat_AsDouble(PyTuple_GET_ITEM(args[5], i));
    for (int i = 0; i < 6; ++i) need[i] = PyObject_IsTrue(PyTuple_GET_ITEM(args[6], i));
    if (PyErr_Occurred()) return nullptr;
    const Tensor &x = s[0], &lb = s[1], &mask = s[2], &ifg = s[3], &xg = s[4], &o = s[5], &attn = s[6], &y = s[7], *nw = s + 8;
    const Tensor& d2 = THPVariable_Unpack(args[0]);
    Tensor grads[12];
    try {
        NoGil nogil;
        OnDevice on(x.get_device());
        // backward() may be called under autocast, which would give the row kernels products of another type than they read
        c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        const auto like = x.options().requires_grad(false);
        const int dt = dtype_of(x.scalar_type());
        const Tensor none, x2 = x.view({m, H});
        std::pair<Tensor, Tensor> products[6];
        auto product = [&](int i, const Tensor& d, const Tensor& yq) { if (need[i]) products[i] = {d, yq}; };
        // The weights' products wait for each other with their operands, 7.75 rows of H an input row at I = 2.75 H.  What nothing reads any more is given
        // back as soon as its last reader is launched, some 10 rows of H, so that a step takes no more memory than with a product at a time.
        // down_proj behind the swiglu: the gradients of gate and up land side by side
        Tensor dz = at::mm(d2, dense(pw[3], like)), dy = at::empty(y.sizes(), like);
        Chained down = chain(CHAIN_SWIGLU, y.narrow(1, 0, I), y.narrow(1, I, I), none, 0.0, {nw[8]}, eps[6], {dz}, none, dy.narrow(1, 0, I), dy.narrow(1, I, I));
        dz.reset();
        product(5, d2, down.y[0]);
        down.y.reset();
        // gate_proj behind mlp_norm, the residual's gradient joining
        Tensor dh = at::mm(dy, dense(pw[2], like));
        Chained gate = chain(CHAIN_RESNORM, attn, x2, nw[1], eps[4], {nw[7]}, eps[5], {dh}, d2, none, none);
        dh.reset();
        product(4, dy, gate.y[0]);
        gate.y.reset();
        dy.reset();
        down.dx.reset();
        // o_proj behind the gated norm: the g columns of the stacked projection's gradient, and the scan's output
        const Tensor& dres = gate.dx;
        Tensor do2 = at::mm(dres, dense(pw[1], like)), difg = at::empty(ifg.sizes(), like), dout = at::empty(o.sizes(), like);
        Chained oc = chain(CHAIN_GATED, ifg.narrow(1, 2 * D, D), o, nw[2], eps[2], {nw[6]}, eps[3], {do2}, none, difg.narrow(1, 2 * D, D), dout);
        do2.reset();
        product(3, dres, oc.y[0]);
        oc.y.reset();
        // scan and gate math
        const auto f32 = like.dtype(at::kFloat);
        const Tensor gates = xg[1].contiguous(), out = o.contiguous();
        Tensor dxs = at::empty({m, D}, like), dgs = at::empty({m, D}, like), ws, dlb, part;
        if (const int64_t bytes = mmf_hgrn_recurrent_bwd_workspace_bytes(b, t, D)) ws = at::empty({bytes / 4}, f32);
        check(mmf_hgrn_recurrent_bwd_split(gates.data_ptr(), out.data_ptr(), dout.data_ptr(), nullptr, dxs.data_ptr(), dgs.data_ptr(), b, t, D, 0, dt, floats(ws),
                                           stream_of(x)),
              "mmf_hgrn_recurrent_bwd_split");
        dout.reset();
        ws.reset();
        if (lb.defined()) {
            dlb = at::empty({D}, f32);
            part = at::empty({mmf_backward_groups(m), D}, f32);
        }
        auto column = [&](const Tensor& a, int64_t j) { return a.narrow(1, j * D, D); };
        const Tensor ii = column(ifg, 0), ff = column(ifg, 1), di = column(difg, 0), df = column(difg, 1);
        check(mmf_hgrn_gate_bwd(ii.data_ptr(), 3 * D, ff.data_ptr(), 3 * D, floats(lb), static_cast<const uint8_t*>(address(mask)), dxs.data_ptr(), dgs.data_ptr(),
                                di.data_ptr(), 3 * D, df.data_ptr(), 3 * D, floats(part), floats(dlb), m, D, dt, stream_of(x)),
              "mmf_hgrn_gate_bwd");
        dxs.reset();
        dgs.reset();
        // i, f, g behind attn_norm: three products, one pass over the rows, the residual's gradient joining
        Chained in;
        {
            const Tensor w3 = dense(pw[0], like), dh3 = at::empty({3, m, H}, like), dhs[3] = {dh3[0], dh3[1], dh3[2]};
            for (int j = 0; j < 3; ++j) {
                Tensor to = dhs[j];
                at::mm_out(to, column(difg, j), w3.narrow(0, j * D, D));
            }
            in = chain(CHAIN_NORM, x2, none, nw[0], eps[0], {nw[3], nw[4], nw[5]}, eps[1], dhs, dres, none, none);
        }
        for (int j = 0; j < 3; ++j) product(j, column(difg, j), in.y[j]);
        const std::vector<Tensor> dw = weight_grads(products);
        grads[0] = in.dx.view(x.sizes());
        grads[1] = dlb;
        grads[2] = in.dw;
        grads[3] = oc.dw;
        grads[4] = gate.dw;
        grads[5] = down.dw;
        for (int i = 0; i < 6; ++i) grads[6 + i] = dw[i];
    } catch (const Failed& f) {
        return failed(f, args[7]);
    }
    PyObject* r = PyTuple_New(12);
    for (int i = 0; r && i < 12; ++i) {
        PyObject* g = Py_None;
        if (grads[i].defined()) g = THPVariable_Wrap(grads[i]);
        else Py_INCREF(g);
        if (!g) { Py_DECREF(r); return nullptr; }
        PyTuple_SET_ITEM(r, i, g);
    }
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
    {"chain_backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(chain_backward)), METH_FASTCALL, nullptr},
    {"dense_weight", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(dense_weight)), METH_FASTCALL, nullptr},
    {"block_backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(block_backward)), METH_FASTCALL, nullptr},
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
