"""Inference of a whole HGRNBitBlock in one native call (mmf_block_forward, csrc/block_forward.hip).

``BlockPlan.of(block)`` lays the pointers of a block's parameters and packed weights out once, in the struct the native
side reads, and remembers what they were taken from.  ``current()`` looks, before every call, whether all of that still
holds: the same modules of the same classes, parameters neither written nor replaced, the same eps, mode, layer index and sizes,
no hook and no patched ``forward`` or ``__call__`` anywhere inside, on a module or on its class -- anything else (and every
block the native call does not cover) goes through the modules.  The results are those of the module path bit for bit: the
same kernels with the same arguments.
"""
import ctypes

import torch
import torch.nn.modules.module as nn_module

from . import _lib as L


class _Block(ctypes.Structure):
    """mmf_block of include/mmf.h."""
    _fields_ = ([(n, ctypes.c_void_p) for n in (
        "attn_norm", "i_norm", "f_norm", "g_proj_norm", "ifg_packed", "ifg_wdeq", "g_norm", "o_norm", "o_packed",
        "o_wdeq", "mlp_norm", "gate_norm", "gate_packed", "gate_wdeq", "down_norm", "down_packed", "down_wdeq")]
        + [(n, ctypes.c_int64) for n in ("o_seg_rows", "gate_seg_rows", "down_seg_rows", "H", "D", "I")]
        + [(n, ctypes.c_float) for n in ("attn_eps", "ifg_eps", "g_eps", "o_eps", "mlp_eps", "gate_eps", "down_eps")]
        + [("dtype", ctypes.c_int), ("weight_dtype", ctypes.c_int)])


def global_hooks():
    """Hooks registered for every module of the process: the module path runs them, the native call does not."""
    return bool(nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks or nn_module._global_backward_hooks
                or nn_module._global_backward_pre_hooks)


AS_DEFINED = {}


def as_defined(cls):
    """Decorator of the classes whose work native calls do in their place: what their forward and __call__ were at the start."""
    AS_DEFINED[cls] = (cls.forward, cls.__call__)
    return cls


def plain(module):
    """Whether a module is one of those classes', unchanged, without a hook or a forward of its own."""
    c = type(module)
    return AS_DEFINED.get(c) == (c.forward, c.__call__) and _untouched(module.__dict__)


def _untouched(d):
    return not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"] or "forward" in d)


class NotCopied:
    """What is laid out once for one module and kept with it: device addresses, the module's own dictionaries, recorded graphs.  A copy
    of the module (deepcopy, or saved whole and loaded) has none of it and makes its own on its first call."""

    def __deepcopy__(self, memo):
        return None

    def __reduce__(self):
        return type(None), ()


class _Structure(NotCopied):
    """The modules of a block and the numbers they carry: what a native call takes for granted besides the parameters.  Nothing here
    leads back to the block itself or its ``__dict__``, which hold this object: a dropped model is freed at once."""

    def __init__(self, block):
        from .attention import HGRNBitAttention
        from .bitlinear import FusedBitLinear
        from .fused_norm_gate import FusedRMSNormSwishGate
        from .layernorm import RMSNorm
        from .modeling_hgrn_bit import HGRNBitBlock, HGRNBitMLP
        self.fits = False
        if type(block) is not HGRNBitBlock:
            return
        attn, mlp = block.attn, block.mlp
        if type(attn) is not HGRNBitAttention or type(mlp) is not HGRNBitMLP or attn.use_short_conv:
            return
        projs = (attn.i_proj, attn.f_proj, attn.g_proj, attn.o_proj, mlp.gate_proj, mlp.down_proj)
        norms = (block.attn_norm, block.mlp_norm, attn.g_norm)
        if (any(type(p) is not FusedBitLinear or p.bias is not None or type(p.norm) is not RMSNorm for p in projs)
                or any(type(n) is not RMSNorm for n in norms[:2]) or type(norms[2]) is not FusedRMSNormSwishGate
                or any(n.weight is None for n in norms) or any(p.norm.weight is None for p in projs)):
            return
        modules = [block, attn, mlp, *norms, *projs, *(p.norm for p in projs)]
        if not all(plain(m) for m in modules):
            return
        H, D, I = attn.hidden_size, attn.input_dim, mlp.intermediate_size
        if (D % 32 or I % 32 or H % 8 or max(H, D, I) > 8192 or attn.num_heads * attn.head_dim != D
                or any(p.run_eps() != projs[0].run_eps() for p in projs[:3])):
            return
        numbers = [(m, "eps") for m in norms + tuple(p.norm for p in projs)] + [(p, "fused_eps") for p in projs] + [(mlp, "intermediate_size")]
        numbers += [(attn, name) for name in ("mode", "layer_idx", "hidden_size", "input_dim", "num_heads", "head_dim", "use_short_conv")]
        self.parameters = [m._parameters for m in modules]
        self.facts = (type(block), block._modules, block._parameters, [(m, type(m), m.__dict__) for m in modules[1:]],
                      [(m._modules, k, c) for m in modules for k, c in m._modules.items()],
                      [(h, k) for h in self.parameters for k, p in h.items() if p is None],
                      [(m.__dict__, name, getattr(m, name)) for m, name in numbers],
                      [(c, *AS_DEFINED[c]) for c in {type(m) for m in modules}])
        self.eps = dict(zip(("attn_eps", "mlp_eps", "g_eps", "ifg_eps", "o_eps", "gate_eps", "down_eps"),
                            [m.eps for m in norms] + [p.run_eps() for p in projs[:1] + projs[3:]]))
        self.attn, self.projs, self.norms = attn, projs, norms
        self.dims, self.heads, self.head_dim, self.mode, self.layer_idx = (H, D, I), attn.num_heads, attn.head_dim, attn.mode, attn.layer_idx
        self.fits = True

    def current(self, block):
        return self.fits and L.native().structure_holds(block, self.facts)

    def norm_weights(self):
        """attn_norm, mlp_norm, g_norm, then the inner norms of i, f, g, o, gate, down."""
        return [m.weight for m in self.norms] + [p.norm.weight for p in self.projs]

    def fits_tensors(self):
        """(dtype, device) of the block's parameters if the native calls take them, else None."""
        H, D, I = self.dims
        ws, nws = [p.weight for p in self.projs], self.norm_weights()
        dt, wdt, dev = ws[0].dtype, nws[0].dtype, nws[0].device
        if (dt not in L._DTYPE_IDS or wdt not in (dt, torch.float32) or dev.type != "cuda"
                or any(w.dtype != dt or w.shape != s for w, s in zip(ws, [(D, H)] * 3 + [(H, D), (2 * I, H), (H, I)]))
                or any(w.dtype != wdt or w.device != dev or not w.is_contiguous() or w.numel() != n
                       for w, n in zip(nws, (H, H, D, H, H, H, D, H, I)))):
            return None
        return dt, dev

    def struct(self, nws, pws, stacked, same, dtype):
        """The native struct over these norm weights and packed weights."""
        H, D, I = self.dims
        o, gate, down = pws[3:]
        return _Block(
            attn_norm=nws[0].data_ptr(), mlp_norm=nws[1].data_ptr(), g_norm=nws[2].data_ptr(), i_norm=nws[3].data_ptr(),
            f_norm=None if same else nws[4].data_ptr(), g_proj_norm=None if same else nws[5].data_ptr(), o_norm=nws[6].data_ptr(),
            gate_norm=nws[7].data_ptr(), down_norm=nws[8].data_ptr(), ifg_packed=stacked.packed.data_ptr(),
            ifg_wdeq=stacked.wdeq.data_ptr(), o_packed=o.packed.data_ptr(), o_wdeq=o.wdeq.data_ptr(), gate_packed=gate.packed.data_ptr(),
            gate_wdeq=gate.wdeq.data_ptr(), down_packed=down.packed.data_ptr(), down_wdeq=down.wdeq.data_ptr(), o_seg_rows=o.seg_rows,
            gate_seg_rows=gate.seg_rows, down_seg_rows=down.seg_rows, H=H, D=D, I=I, dtype=L.dtype_id(dtype),
            weight_dtype=L.dtype_id(nws[0].dtype), **self.eps)


def _structure(block):
    s = block.__dict__.get("_native_structure")
    if s is None or not s.current(block):
        s = block.__dict__["_native_structure"] = _Structure(block)
    return s


class BlockPlan(NotCopied):
    """The native form of one block for inference: ``None`` from ``of`` where there is none."""

    @classmethod
    def of(cls, block):
        plan = block.__dict__.get("_native_plan")
        if plan is None or not plan.current(block):
            plan = block.__dict__["_native_plan"] = cls(block)
        return plan if plan.fits else None

    def __init__(self, block):
        self.fits = False
        s = self.structure = _structure(block)
        where = s.fits_tensors() if s.fits else None
        if where is None:
            return
        self.params = [(h, k, p, p._version, p.data_ptr()) for h in s.parameters for k, p in h.items() if p is not None]
        self.dtype, self.device = where
        nws, pws = s.norm_weights(), [p.packed_weight() for p in s.projs]
        if any(pw.packed.device != self.device for pw in pws):
            return
        self.packed = [(p._pack, pw) for p, pw in zip(s.projs, pws)]
        self.stacked = s.attn._stacked_weight()
        same = all(torch.equal(nws[3], w) for w in nws[4:6])
        self.native = s.struct(nws, pws, self.stacked, same, self.dtype)
        self.ref = ctypes.addressof(self.native)
        self.dims, self.heads, self.head_dim, self.mode, self.layer_idx = s.dims, s.heads, s.head_dim, s.mode, s.layer_idx
        self.H, self.D = s.dims[:2]
        self.fits = True

    def current(self, block):
        if not (self.fits and self.structure.current(block)):
            return False
        if not L.native().parameters_hold(self.params):
            return False
        for pack, pw in self.packed:
            if pack.pw is not pw:
                return False
        return True


class TrainPlan:
    """One training forward of a block: its struct over today's parameters (an optimizer step changes them all)."""

    @classmethod
    def of(cls, block, x):
        s = _structure(block)
        if not s.fits or max(s.dims[:2]) > 4096 or s.mode != "fused_recurrent":
            return None
        where = s.fits_tensors()
        if where is None or where != (x.dtype, x.device) or any(p.weight.is_meta for p in s.projs):
            return None
        return cls(s, where[0])

    def __init__(self, s, dtype):
        self.dims, self.layer_idx = s.dims, s.layer_idx
        self.pws = [p.packed_weight() for p in s.projs]
        self.stacked = s.attn._stacked_weight()
        self.eps = s.eps
        self.norm_params = s.norm_weights()
        self.weight_params = [p.weight for p in s.projs]
        self.native = s.struct(self.norm_params, self.pws, self.stacked, False, dtype)
        self.ref = ctypes.addressof(self.native)


def workspace(plan, rows):
    lib = L.load()
    if lib.mmf_block_struct_bytes() != ctypes.sizeof(_Block):
        raise L.MMFError("block.py and include/mmf.h disagree about mmf_block")
    # torch hands out 512-byte aligned blocks
    return torch.empty(lib.mmf_block_workspace_bytes(plan.ref, rows), dtype=torch.uint8, device=plan.device)


def forward(plan, x, out, b, t, lower_bound, mask, h0, ht, ws, stream):
    """out = block(x); all tensors checked by the caller.  h0 / ht: state addresses or None."""
    L.check(L.load().mmf_block_forward(plan.ref, x, out, b, t, lower_bound, mask, h0, ht, ws, stream), "mmf_block_forward")
