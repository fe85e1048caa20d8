"""Inference of a whole HGRNBitBlock in one native call (mmf_block_forward, csrc/block_forward.hip).

``BlockPlan.of(block)`` lays the pointers of a block's parameters and packed weights out once, in the struct the native
side reads, and remembers what they were taken from.  ``current()`` looks, before every call, whether all of that still
holds: the same modules, parameters neither written nor replaced, the same eps, no hook and no patched ``forward`` anywhere
inside -- anything else (and every block the native call does not cover) goes through the modules as before.  The
results are those of the module path bit for bit: the same kernels with the same arguments.
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
    return bool(nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks)


def hook_free(module):
    d = module.__dict__
    return not (d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d)


class BlockPlan:
    """The native form of one block: ``None`` from ``of`` where there is none."""

    @classmethod
    def of(cls, block):
        plan = block.__dict__.get("_native_plan")
        if plan is not None and plan.current():
            return plan if plan.fits else None
        plan = block.__dict__["_native_plan"] = cls(block)
        return plan if plan.fits else None

    def __init__(self, block):
        from .attention import HGRNBitAttention
        from .bitlinear import FusedBitLinear
        from .fused_norm_gate import FusedRMSNormSwishGate
        from .layernorm import RMSNorm
        from .modeling_hgrn_bit import HGRNBitBlock, HGRNBitMLP
        self.fits = False
        self.modules = list(block.modules())
        self.dicts = [m.__dict__ for m in self.modules]
        # what the plan depends on: children, parameters (object, version, address), the numbers it copies
        self.children = [(d["_modules"], k, c) for d in self.dicts for k, c in d["_modules"].items()]
        self.params = [(d["_parameters"], k, p, p._version, p.data_ptr()) for d in self.dicts
                       for k, p in d["_parameters"].items() if p is not None]
        self.absent = [(d["_parameters"], k) for d in self.dicts for k, p in d["_parameters"].items() if p is None]
        self.numbers, self.packed = [], []
        attn, mlp = block.attn, block.mlp
        if (type(block) is not HGRNBitBlock or type(attn) is not HGRNBitAttention or type(mlp) is not HGRNBitMLP
                or attn.use_short_conv or any("forward" in d for d in self.dicts)):
            return
        projs = (attn.i_proj, attn.f_proj, attn.g_proj, attn.o_proj, mlp.gate_proj, mlp.down_proj)
        norms = (block.attn_norm, block.mlp_norm)
        if (any(type(p) is not FusedBitLinear or p.bias is not None or type(p.norm) is not RMSNorm for p in projs)
                or any(type(n) is not RMSNorm for n in norms) or type(attn.g_norm) is not FusedRMSNormSwishGate):
            return
        norm_ws = [m.weight for m in norms + (attn.g_norm,)] + [p.norm.weight for p in projs]
        if any(w is None or not w.is_cuda or not w.is_contiguous() or w.dtype != norm_ws[0].dtype for w in norm_ws):
            return
        dt, wdt, dev = projs[0].weight.dtype, norm_ws[0].dtype, norm_ws[0].device
        H, D, I = attn.hidden_size, attn.input_dim, mlp.intermediate_size
        shapes = [(D, H)] * 3 + [(H, D), (2 * I, H), (H, I)]
        if (dt not in L._DTYPE_IDS or any(p.weight.dtype != dt or tuple(p.weight.shape) != s for p, s in zip(projs, shapes))
                or wdt not in (dt, torch.float32) or any(w.device != dev for w in norm_ws)
                or [w.numel() for w in norm_ws] != [H, H, D, H, H, H, D, H, I]
                or D % 32 or I % 32 or H % 8 or max(H, D, I) > 8192 or attn.num_heads * attn.head_dim != D):
            return
        eps = [block.attn_norm.eps, projs[0].run_eps(), attn.g_norm.eps, projs[3].run_eps(), block.mlp_norm.eps,
               projs[4].run_eps(), projs[5].run_eps()]
        if any(p.run_eps() != projs[0].run_eps() for p in projs[:3]):
            return
        same = all(torch.equal(projs[0].norm.weight, p.norm.weight) for p in projs[1:3])
        pws = [p.packed_weight() for p in projs]
        if any(pw.packed.device != dev for pw in pws):
            return
        ifg = attn._stacked_weight()
        self.numbers = ([(m, "eps", m.eps) for m in norms + (attn.g_norm,) + tuple(p.norm for p in projs)]
                        + [(p, "fused_eps", p.fused_eps) for p in projs])
        self.packed = [(p._pack, pw) for p, pw in zip(projs, pws)]
        self.keep = ifg
        self.dtype, self.device, self.H, self.D, self.I = dt, dev, H, D, I
        self.dims, self.heads, self.head_dim, self.mode = (H, D, I), attn.num_heads, attn.head_dim, attn.mode
        o, gate, down = pws[3:]
        nw = [w.data_ptr() for w in norm_ws]
        self.struct = _Block(
            attn_norm=nw[0], i_norm=nw[3], f_norm=None if same else nw[4], g_proj_norm=None if same else nw[5],
            ifg_packed=ifg.packed.data_ptr(), ifg_wdeq=ifg.wdeq.data_ptr(), g_norm=nw[2], o_norm=nw[6], o_packed=o.packed.data_ptr(),
            o_wdeq=o.wdeq.data_ptr(), mlp_norm=nw[1], gate_norm=nw[7], gate_packed=gate.packed.data_ptr(),
            gate_wdeq=gate.wdeq.data_ptr(), down_norm=nw[8], down_packed=down.packed.data_ptr(), down_wdeq=down.wdeq.data_ptr(),
            o_seg_rows=o.seg_rows, gate_seg_rows=gate.seg_rows, down_seg_rows=down.seg_rows, H=H, D=D, I=I,
            attn_eps=eps[0], ifg_eps=eps[1], g_eps=eps[2], o_eps=eps[3], mlp_eps=eps[4], gate_eps=eps[5], down_eps=eps[6],
            dtype=L.dtype_id(dt), weight_dtype=L.dtype_id(wdt))
        self.ref = ctypes.addressof(self.struct)
        self.layer_idx = attn.layer_idx
        self.fits = True

    def current(self):
        for d in self.dicts:
            if d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d:
                return False
        for d, k, p, version, address in self.params:
            if d.get(k) is not p or p._version != version or p.data_ptr() != address:
                return False
        for d, k, c in self.children:
            if d.get(k) is not c:
                return False
        for d, k in self.absent:
            if d.get(k) is not None:
                return False
        for m, k, v in self.numbers:
            if getattr(m, k) != v:
                return False
        for pack, pw in self.packed:
            if pack.pw is not pw:
                return False
        return True


def workspace(plan, rows):
    lib = L.load()
    if lib.mmf_block_struct_bytes() != ctypes.sizeof(_Block):
        raise L.MMFError("block.py and include/mmf.h disagree about mmf_block")
    # torch hands out 512-byte aligned blocks
    return torch.empty(lib.mmf_block_workspace_bytes(plan.ref, rows), dtype=torch.uint8, device=plan.device)


def forward(plan, x, out, b, t, lower_bound, mask, h0, ht, ws, stream):
    """out = block(x); all tensors checked by the caller.  h0 / ht: state addresses or None."""
    L.check(L.load().mmf_block_forward(plan.ref, x, out, b, t, lower_bound, mask, h0, ht, ws, stream), "mmf_block_forward")
