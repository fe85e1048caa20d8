"""Training side: torch.autograd.Functions over the HIP forward and backward kernels.

Each Function mirrors one of the reference's autograd Functions:
  BitLinearFn              LayerNormLinearQuantFn        mmfreelm/ops/fusedbitnet.py:416-510
  RMSNormFn                LayerNormFn (RMS form)        mmfreelm/modules/layernorm.py:445-531
  RMSNormSwishGateFn       LayerNormFn (gated)           mmfreelm/modules/fused_norm_gate.py:420-500
  SwiGLUFn                 SwiGLUFunction                mmfreelm/modules/activations.py:143-175
  BlockFn, NormHeadFn      a whole block / final norm + head of mmfreelm/models/hgrn_bit/modeling_hgrn_bit.py:97-111, 262, 386
  HGRNGateFn               the elementwise ops of mmfreelm/layers/hgrn_bit.py:113-120, differentiated as one op
  CrossEntropyFn           CrossEntropyLossFunction      mmfreelm/modules/fused_cross_entropy.py:163-310

The forward values are those of the inference kernels (same launches); the backward kernels live in csrc/backward.hip,
csrc/backward_block.hip (a block's row kernels) and csrc/hgrn_block.hip (the scans).
The two dense products of a BitLinear's backward (dout @ W_q and dout^T @ y_q, fusedbitnet.py:474, :498) are plain
library GEMMs (torch.matmul).  Modules pick these Functions when gradients are enabled and an input or parameter
requires one (`needs_grad`); otherwise they keep the fused inference launches.  The scans differentiate in native code
(csrc/torch_ops.cpp).
"""
import ctypes

import torch

from . import _lib as L
from . import functional as F_


def needs_grad(*tensors) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


def module_needs_grad(module, *inputs) -> bool:
    """The rule every module uses to pick the differentiable path: gradients are enabled and an input or one of the module's
    parameters requires one -- whatever module.training says (the reference differentiates in eval mode too)."""
    return torch.is_grad_enabled() and (any(t is not None and t.requires_grad for t in inputs)
                                        or any(p.requires_grad for p in module.parameters()))


def _2d(t):
    return t.reshape(-1, t.shape[-1])


def _rows_ld(t):
    """[rows, K] view and its row stride; copies only if the last dimension is strided."""
    t2 = _2d(t)
    if t2.stride(-1) != 1 or (t2.shape[0] > 1 and t2.stride(0) < t2.shape[1]):
        t2 = t2.contiguous()
    return t2, (t2.stride(0) if t2.shape[0] > 1 else t2.shape[1])


def _norm_bwd(mode, xs, gate, weight, dy, dres, eps, want_y=False):
    """Launch mmf_rmsnorm_bwd; returns (dx, dgate, y_quant, dweight)."""
    lib = L.load()
    dev = xs.device
    x2, ldx = _rows_ld(xs)
    dy2, lddy = _rows_ld(dy if dy.dtype == x2.dtype else dy.to(x2.dtype))
    m, k = x2.shape
    g2, ldg = _rows_ld(gate) if gate is not None else (None, 0)
    dr2 = _2d(dres).to(x2.dtype).contiguous() if dres is not None else None
    dx = torch.empty(m, k, dtype=x2.dtype, device=dev)
    dgate = torch.empty(m, k, dtype=x2.dtype, device=dev) if mode == 1 else None
    yq = torch.empty(m, k, dtype=x2.dtype, device=dev) if want_y else None
    w = F_.vector(weight, k, "norm weight")
    if w is not None and w.dtype not in (torch.float32, x2.dtype):
        w = w.float()
    dw = torch.empty_like(w) if w is not None else None
    part = torch.empty(lib.mmf_backward_groups(m), k, dtype=torch.float32, device=dev) if w is not None else None
    with L.on(dev):
        L.check(lib.mmf_rmsnorm_bwd(mode, x2.data_ptr(), ldx, L.ptr(g2), ldg, L.ptr(w), dy2.data_ptr(), lddy, L.ptr(dr2),
                                    dx.data_ptr(), L.ptr(dgate), L.ptr(yq), L.ptr(part), L.ptr(dw), m, k, eps,
                                    L.dtype_id(x2.dtype), L.dtype_id(w.dtype) if w is not None else 0, L.stream()),
                "mmf_rmsnorm_bwd")
    if dw is not None and weight is not None and dw.dtype != weight.dtype:
        dw = dw.to(weight.dtype)
    return dx, dgate, yq, dw


class RMSNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, residual, eps, prenorm, residual_in_fp32):
        with torch.no_grad():
            if residual is not None or prenorm:
                y, res_out = F_.rmsnorm(x, weight, residual=residual, eps=eps, prenorm=True, residual_in_fp32=residual_in_fp32)
            else:
                y, res_out = F_.rmsnorm(x, weight, eps=eps), x
        ctx.save_for_backward(res_out, weight)
        ctx.eps, ctx.has_res, ctx.prenorm, ctx.x_dtype, ctx.shape = eps, residual is not None, prenorm, x.dtype, x.shape
        ctx.res_dtype = residual.dtype if residual is not None else None
        return (y, res_out) if prenorm else y

    @staticmethod
    def backward(ctx, dy, *rest):
        xs, weight = ctx.saved_tensors
        dres = rest[0] if (ctx.prenorm and rest and rest[0] is not None) else None
        dx, _, _, dw = _norm_bwd(0, xs, None, weight, dy.contiguous(), dres, ctx.eps)
        dx = dx.reshape(ctx.shape)
        dres_in = dx.to(ctx.res_dtype) if ctx.has_res else None
        return dx.to(ctx.x_dtype), dw, dres_in, None, None, None


class RMSNormSwishGateFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, o, weight, eps):
        with torch.no_grad():
            y = F_.rmsnorm_swishgate(x, o, weight, eps=eps)
        ctx.save_for_backward(x, o, weight)
        ctx.eps = eps
        return y

    @staticmethod
    def backward(ctx, dy):
        x, o, weight = ctx.saved_tensors
        dx, do, _, dw = _norm_bwd(1, x, o, weight, dy.contiguous(), None, ctx.eps)
        return dx.reshape(x.shape), do.reshape(o.shape), dw, None


class BitLinearFn(torch.autograd.Function):
    """RMSNorm -> int8 absmax quantiser -> ternary weights, straight-through gradients (fusedbitnet.py:416-510)."""

    @staticmethod
    def forward(ctx, x, norm_weight, weight, bias, eps, residual, prenorm, residual_in_fp32, pw):
        with torch.no_grad():
            if pw is None:
                pw = F_.ternarize_pack(weight)
            if residual is not None or prenorm:
                out, res_out = F_.bitlinear(x, norm_weight, pw, bias=bias, eps=eps, residual=residual, prenorm=True,
                                            residual_in_fp32=residual_in_fp32)
            else:
                out, res_out = F_.bitlinear(x, norm_weight, pw, bias=bias, eps=eps), x
        ctx.save_for_backward(res_out, norm_weight)
        ctx.pw, ctx.eps, ctx.has_res, ctx.prenorm, ctx.has_bias = pw, eps, residual is not None, prenorm, bias is not None
        ctx.w_dtype, ctx.x_dtype, ctx.shape = weight.dtype, x.dtype, x.shape
        ctx.res_dtype = residual.dtype if residual is not None else None
        ctx.bias_dtype = bias.dtype if bias is not None else None
        return (out, res_out) if prenorm else out

    @staticmethod
    def backward(ctx, dout, *rest):
        xs, norm_weight = ctx.saved_tensors
        pw = ctx.pw
        dres = rest[0] if (ctx.prenorm and rest and rest[0] is not None) else None
        d2 = _2d(dout).contiguous()
        # de-quantised ternary weights [N, K] in the activation dtype: t * wdeq
        wq = F_.unpack_ternary(pw).to(d2.dtype) * pw.wdeq.to(d2.dtype)
        dy = d2 @ wq                                                  # fusedbitnet.py:474
        dx, _, yq, dnw = _norm_bwd(2, xs, None, norm_weight, dy, dres, ctx.eps, want_y=True)
        dw = (d2.t() @ yq.to(d2.dtype)).to(ctx.w_dtype)              # fusedbitnet.py:498
        dbias = d2.sum(0).to(ctx.bias_dtype) if ctx.has_bias else None
        dx = dx.reshape(ctx.shape)
        dres_in = dx.to(ctx.res_dtype) if ctx.has_res else None
        return dx.to(ctx.x_dtype), dnw, dw, dbias, None, dres_in, None, None, None


class SwiGLUFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, y):
        with torch.no_grad():
            out = F_.swiglu(x, y)
        ctx.save_for_backward(x, y)
        return out

    @staticmethod
    def backward(ctx, g):
        x, y = ctx.saved_tensors
        lib = L.load()
        x2, ldx = _rows_ld(x)
        y2, ldy = _rows_ld(y)
        g2, ldg = _rows_ld(g)
        rows, cols = x2.shape
        dx = torch.empty(rows, cols, dtype=x.dtype, device=x.device)
        dy = torch.empty(rows, cols, dtype=x.dtype, device=x.device)
        with L.on(x.device):
            L.check(lib.mmf_swiglu_bwd(x2.data_ptr(), ldx, y2.data_ptr(), ldy, g2.data_ptr(), ldg, dx.data_ptr(), cols,
                                       dy.data_ptr(), cols, rows, cols, L.dtype_id(x.dtype), L.stream()), "mmf_swiglu_bwd")
        return dx.reshape(x.shape), dy.reshape(y.shape)


class HGRNGateFn(torch.autograd.Function):
    """(i, f) -> (x, g) of mmfreelm/layers/hgrn_bit.py:113-120 as one differentiable op."""

    @staticmethod
    def forward(ctx, i, f, lower_bound, mask):
        with torch.no_grad():
            x, g = F_.hgrn_gate(i, f, lower_bound, mask)
        ctx.save_for_backward(i, f, lower_bound, mask)
        return x, g

    @staticmethod
    def backward(ctx, gx, gg):
        i, f, lb, mask = ctx.saved_tensors
        lib = L.load()
        dev = i.device
        d = i.shape[-1]
        i2, ldi = _rows_ld(i)
        f2, ldf = _rows_ld(f)
        rows = i2.shape[0]
        gx2 = _2d(gx).to(i.dtype).contiguous() if gx is not None else torch.zeros(rows, d, dtype=i.dtype, device=dev)
        gg2 = _2d(gg).to(i.dtype).contiguous() if gg is not None else torch.zeros(rows, d, dtype=i.dtype, device=dev)
        di = torch.empty(rows, d, dtype=i.dtype, device=dev)
        df = torch.empty(rows, d, dtype=i.dtype, device=dev)
        lbf = F_.lower_bound_row(lb, d)
        dlb = torch.empty(d, dtype=torch.float32, device=dev) if lb is not None else None
        part = torch.empty(lib.mmf_backward_groups(rows), d, dtype=torch.float32, device=dev) if lb is not None else None
        mk = F_._mask_rows(mask, rows, dev) if mask is not None else None
        with L.on(dev):
            L.check(lib.mmf_hgrn_gate_bwd(i2.data_ptr(), ldi, f2.data_ptr(), ldf, L.ptr(lbf), L.ptr(mk), gx2.data_ptr(),
                                          gg2.data_ptr(), di.data_ptr(), d, df.data_ptr(), d, L.ptr(part), L.ptr(dlb), rows, d,
                                          L.dtype_id(i.dtype), L.stream()), "mmf_hgrn_gate_bwd")
        return di.reshape(i.shape), df.reshape(f.shape), (dlb.to(lb.dtype) if lb is not None else None), None


CHAIN_NORM, CHAIN_GATED, CHAIN_SWIGLU, CHAIN_RESNORM = 0, 1, 2, 3


def _chain_bwd(kind, x, aux, w1, eps1, w2, eps2, dy, dres=None, dx=None, daux=None):
    """mmf_chain_bwd over [M, K] operands (column slices keep their row stride; dy [norms, M, K]):
    (dx, daux, y_quant [norms, M, K], weight gradients [(w1) + norms, K])."""
    dx, y, dw = L.native().chain_backward(kind, x, aux, w1, eps1, tuple(w2), eps2, tuple(dy), dres, dx, daux, L.check)
    return dx, daux, y, dw


def _dense_weight(pw, dtype):
    """The dense ternary weights [N, K] for dout @ W_q."""
    return L.native().dense_weight(pw.packed, pw.wdeq, pw.seg_rows, pw.n, pw.k, dtype, L.check)


def _turns(dout, y):
    """Whether mmf_weight_grad takes a product: rows of whole, aligned 16-byte pieces."""
    whole = 16 // y.element_size()
    return y.dtype in (torch.float32, torch.bfloat16, torch.float16) and dout.dtype == y.dtype and 0 < len(dout) <= 0x7fffffff and all(
        t.stride(1) == 1 and t.shape[1] > 0 and t.shape[1] % whole == 0 and t.stride(0) % whole == 0 and t.shape[1] <= t.stride(0) <= 1 << 24
        and t.data_ptr() % 16 == 0 for t in (dout, y))


def _turned_products(pairs):
    """[dout^T @ y] of [M, N] gradients and [M, K] inputs over the same M rows, at most eight, in one launch."""
    lib, n, m = L.load(), len(pairs), pairs[0][0].shape[0]
    ptrs, ints = ctypes.c_void_p * n, ctypes.c_int64 * n
    ns, ks = ints(*[d.shape[1] for d, _ in pairs]), ints(*[y.shape[1] for _, y in pairs])
    out = [torch.empty(d.shape[1], y.shape[1], dtype=y.dtype, device=y.device) for d, y in pairs]
    size = lib.mmf_weight_grad_workspace_bytes(n, ns, ks, m, L.dtype_id(out[0].dtype))
    ws = torch.empty(size, dtype=torch.uint8, device=out[0].device) if size else None
    L.check(lib.mmf_weight_grad(n, ptrs(*[d.data_ptr() for d, _ in pairs]), ints(*[d.stride(0) for d, _ in pairs]),
                                ptrs(*[y.data_ptr() for _, y in pairs]), ints(*[y.stride(0) for _, y in pairs]),
                                ptrs(*[o.data_ptr() for o in out]), ns, ks, m, L.dtype_id(out[0].dtype), L.ptr(ws), L.stream()), "mmf_weight_grad")
    return out


def _weight_grad(dout, y):
    """dout^T @ y_q of [M, N] gradients and [M, K] de-quantised inputs.

    For as many outputs as a vocabulary the inputs are stored [K, M] first, contiguous along the contraction, where the library's kernels
    run at a higher rate then: rows a multiple of 64, from 3000 on of 8.  bf16, us, as they are / transposed: 8192 x 1024 -> 32000 488 / 428,
    8192 x 2048 1097 / 816, 3072 x 2048 10 % less, 1024 x 2048 152 / 131, 5000 rows 7 % less; 1056 rows 20 % more, 2016 5 % more, 2002 and 3001, which
    are no multiple of 8 (the transposition moves single elements), 0 to 7 % more; the same for 16384 to 50304 outputs and in fp16.  For fewer outputs the
    transposition, 4 bytes an element, costs more of the product (11264: 4 %) than it gives there (-5 to 12 %).
    Other rows, from 600 on, take mmf_weight_grad: 2048 -> 32000 666 rows 128 us by the library, 105 by it, 2002 rows 266 and 237 (1024 wide 69 and 54, 138 and
    121); 512 rows 88 and 89.  Where the transposition pays it is 4 to 8 % behind (8192 rows 878 us)."""
    m, k = y.shape
    if y.element_size() == 2 and dout.shape[1] >= 16384 and y.is_contiguous():
        if 1024 <= m <= 4194240 and (m % 64 == 0 if m < 3000 else m % 8 == 0):
            yt = torch.empty(k, m, dtype=y.dtype, device=y.device)
            L.check(L.load().mmf_transpose16(y.data_ptr(), m, k, yt.data_ptr(), L.stream()), "mmf_transpose16")
            y = yt.t()
        elif m >= 600 and _turns(dout, y):
            return _turned_products([(dout, y)])[0]
    return dout.t() @ y


class BlockFn(torch.autograd.Function):
    """A whole HGRNBitBlock (mmfreelm/models/hgrn_bit/modeling_hgrn_bit.py:97-111) as one differentiable op.

    The forward is one native call that gives the bits of the op-by-op composition.  The backward runs the same dense
    products as that composition's (dout @ W_q and dout^T @ y_q per BitLinear) and one row kernel between them where the
    composition had a norm behind a norm, three norms added up, or sliced tensors to put together; it is native too.
    ``params``: the nine norm weights (block.py's order), then the six BitLinear weights i, f, g, o, gate, down."""

    @staticmethod
    def forward(ctx, plan, x, lower_bound, mask, *params):
        lib = L.load()
        H, D, I = plan.dims
        b, t, _ = x.shape
        m = b * t
        x = x.contiguous()
        dev, dt = x.device, x.dtype
        with L.on(dev):
            empty = lambda *shape: torch.empty(*shape, dtype=dt, device=dev)
            out, ifg, xg, o, attn, y = torch.empty_like(x), empty(m, 3 * D), empty(2, m, D), empty(m, D), empty(m, H), empty(m, 2 * I)
            lb = F_.lower_bound_row(lower_bound, D)
            mk = F_._mask_rows(mask, m, dev)
            ws = torch.empty(lib.mmf_block_train_workspace_bytes(plan.ref, m), dtype=torch.uint8, device=dev)
            L.check(lib.mmf_block_train_forward(plan.ref, x.data_ptr(), out.data_ptr(), ifg.data_ptr(), xg.data_ptr(), o.data_ptr(),
                                                attn.data_ptr(), y.data_ptr(), b, t, L.ptr(lb), L.ptr(mk), ws.data_ptr(), L.stream()),
                    "mmf_block_train_forward")
        ctx.save_for_backward(x, lb, mk, ifg, xg, o, attn, y, *params[:9])
        ctx.plan, ctx.lb_dtype = plan, lower_bound.dtype if lower_bound is not None else None
        return out

    @staticmethod
    def backward(ctx, dout):
        x, lb, mk, ifg, xg, o, attn, y, *nw = ctx.saved_tensors
        plan, eps = ctx.plan, ctx.plan.eps
        b, t, H = x.shape
        d2 = dout.to(x.dtype).reshape(b * t, H).contiguous()
        packed = tuple((pw.packed, pw.wdeq, pw.seg_rows, pw.n, pw.k) for pw in (plan.stacked, *plan.pws[3:]))
        dx, dlb, ifg_n, o_n, gate_n, down_n, *d_weights = L.native().block_backward(
            d2, (b, t), plan.dims, (x, lb, mk, ifg, xg, o, attn, y, *nw), packed,
            tuple(float(eps[k]) for k in ("attn_eps", "ifg_eps", "g_eps", "o_eps", "mlp_eps", "gate_eps", "down_eps")), ctx.needs_input_grad[13:19], L.check)
        grads = [ifg_n[0], gate_n[0], o_n[0], ifg_n[1], ifg_n[2], ifg_n[3], o_n[1], gate_n[1], down_n[0]]
        if dlb is not None:
            dlb = dlb.to(ctx.lb_dtype)
        return (None, dx, dlb, None, *grads, *d_weights)


class NormHeadFn(torch.autograd.Function):
    """The final norm and the head's BitLinear (mmfreelm/models/hgrn_bit/modeling_hgrn_bit.py:262, 386) as one op."""

    @staticmethod
    def forward(ctx, x, norm_weight, head_norm_weight, weight, pw, eps1, eps2):
        with torch.no_grad():
            out = F_.bitlinear(x, head_norm_weight, pw, eps=eps2, prologue=("norm", norm_weight, eps1))
        ctx.save_for_backward(x, norm_weight, head_norm_weight)
        ctx.pw, ctx.eps1, ctx.eps2 = pw, eps1, eps2
        return out

    @staticmethod
    def backward(ctx, dout):
        x, norm_weight, head_norm_weight = ctx.saved_tensors
        with L.on(x.device):
            x2, d2 = _2d(x).contiguous(), _2d(dout).to(x.dtype).contiguous()
            dh = (d2 @ _dense_weight(ctx.pw, x.dtype)).to(x.dtype)    # (another type under autocast)
            dx, _, yq, dw = _chain_bwd(CHAIN_NORM, x2, None, norm_weight, ctx.eps1, [head_norm_weight], ctx.eps2, [dh])
            d_weight = _weight_grad(d2, yq[0]) if ctx.needs_input_grad[3] else None
        return dx.view(x.shape), dw[0], dw[1], d_weight, None, None, None


class CrossEntropyFn(torch.autograd.Function):
    """Per-row losses (and z-losses) of [rows, V] logits; mmfreelm/modules/fused_cross_entropy.py:163-310 on one device."""

    @staticmethod
    def forward(ctx, logits, labels, smoothing, logit_scale, lse_square_scale, ignore_index, inplace_backward):
        lib = L.load()
        dev = L.require_gpu(logits, labels)
        if logits.dim() != 2 or labels.shape != (logits.shape[0],):
            raise ValueError("logits [rows, V] and one label per row")
        lg = logits if logits.stride(-1) == 1 else logits.contiguous()
        lab = labels.to(torch.int64).contiguous()
        rows, v = lg.shape
        loss = torch.empty(rows, dtype=torch.float32, device=dev)
        lse = torch.empty(rows, dtype=torch.float32, device=dev)
        z = torch.empty(rows, dtype=torch.float32, device=dev)
        with L.on(dev):
            L.check(lib.mmf_cross_entropy_train_fwd(lg.data_ptr(), lg.stride(0), lab.data_ptr(), int(ignore_index), float(smoothing),
                                                    float(logit_scale), float(lse_square_scale), loss.data_ptr(), lse.data_ptr(),
                                                    z.data_ptr(), rows, v, L.dtype_id(lg.dtype), L.stream()),
                    "mmf_cross_entropy_train_fwd")
        ctx.save_for_backward(lg, lab, lse)
        ctx.args = (float(smoothing), float(logit_scale), float(lse_square_scale), int(ignore_index), bool(inplace_backward))
        ctx.mark_non_differentiable(z)
        return loss, z

    @staticmethod
    def backward(ctx, dloss, dz=None):
        lg, lab, lse = ctx.saved_tensors
        smoothing, logit_scale, lse_square_scale, ignore_index, inplace = ctx.args
        lib = L.load()
        rows, v = lg.shape
        dlogits = lg if inplace else torch.empty_like(lg)
        dl = dloss.to(torch.float32).contiguous()
        with L.on(lg.device):
            L.check(lib.mmf_cross_entropy_train_bwd(lg.data_ptr(), lg.stride(0), lab.data_ptr(), ignore_index, lse.data_ptr(),
                                                    dl.data_ptr(), smoothing, logit_scale, lse_square_scale, dlogits.data_ptr(),
                                                    dlogits.stride(0), rows, v, L.dtype_id(lg.dtype), L.stream()),
                    "mmf_cross_entropy_train_bwd")
        return dlogits, None, None, None, None, None, None


class FusedCrossEntropyLoss(torch.nn.Module):
    """mmfreelm/modules/fused_cross_entropy.py:323-398 (one device: no process_group)."""

    def __init__(self, ignore_index=-100, reduction="mean", label_smoothing=0.0, logit_scale=1.0, lse_square_scale=0.0,
                 inplace_backward=False, process_group=None, return_z_loss=False):
        super().__init__()
        if reduction not in ("mean", "none", "sum"):
            raise NotImplementedError("Only support reduction = 'mean' or 'none' or 'sum'")
        if process_group is not None:
            raise NotImplementedError("the vocabulary-parallel loss needs a process group; this build runs on one GPU")
        self.ignore_index, self.reduction, self.label_smoothing = ignore_index, reduction, label_smoothing
        self.logit_scale, self.lse_square_scale = logit_scale, lse_square_scale
        self.inplace_backward, self.return_z_loss = inplace_backward, return_z_loss

    def forward(self, input, target):
        loss, z_loss = CrossEntropyFn.apply(input, target, self.label_smoothing, self.logit_scale, self.lse_square_scale,
                                            self.ignore_index, self.inplace_backward)
        if self.reduction == "mean":
            n = (target != self.ignore_index).sum()
            loss, z_loss = loss.sum() / n, z_loss.sum() / n
        elif self.reduction == "sum":
            loss, z_loss = loss.sum(), z_loss.sum()
        return (loss, z_loss) if self.return_z_loss else loss


class ShortConvFn(torch.autograd.Function):
    """ShortConvolution.forward over whole sequences (mmfreelm/modules/convolution.py:98-131) as one differentiable op."""

    @staticmethod
    def forward(ctx, x, weight, bias, activation):
        with torch.no_grad():
            y = F_.short_conv(x, weight, bias, activation)
        ctx.save_for_backward(x, weight, bias)
        ctx.activation = activation
        return y

    @staticmethod
    def backward(ctx, g):
        x, weight, bias = ctx.saved_tensors
        dx, dw, db = F_.short_conv_bwd(x, weight, bias, g, ctx.activation)
        dweight = dw.reshape(weight.shape).to(weight.dtype) if ctx.needs_input_grad[1] else None
        dbias = db.to(bias.dtype) if (bias is not None and ctx.needs_input_grad[2]) else None
        return dx, dweight, dbias, None
