"""Whole-model single-token decode step as one launch or one HIP graph.

At batch 1 the whole step -- embedding row, the 4L fused BitLinears of the layers, final norm and lm_head, argmax -- is ONE
persistent launch (mmf_decode_layers_norms: resident workgroups hand activations to each other as tagged words), launched
directly, where the model fits it; a step that samples is followed by the launch of its draw.

The module path (HGRNBitForCausalLM.forward with T = 1) issues the same kernels through
nn.Module calls and fresh output tensors; at batch 1 that host work dwarfs the ~40 us the
weights take to stream.  DecodeEngine lays the step out once over static buffers; beyond batch 1 (or that
launch's limits) it records it into a graph (torch.cuda.CUDAGraph = hipGraph) and replays it per token: embedding gather ->
L x [RMSNorm, i/f/g BitLinear, gate + recurrence step, gated norm, o_proj BitLinear,
residual RMSNorm, gate_proj BitLinear, swiglu, down_proj BitLinear (+residual)] -> final
norm -> lm_head BitLinear -> argmax or draw.  The last writes the token buffer the next step's
embedding reads, so consecutive steps need no host round trip; the tokens fed are recorded by the step itself.

Every launch is the same C-ABI call with the same arithmetic as the module path, so the two
produce identical bits (tests/test_gpu_model.py checks that).
"""
import ctypes
import struct
import warnings
from typing import List, Optional

import torch

from . import _lib as L
from . import functional as F_
from .block import NotCopied


class _Phase(ctypes.Structure):
    """One fused BitLinear of mmf_decode_layers' device table (include/mmf.h)."""
    _fields_ = [("w1", ctypes.c_void_p), ("norm_w", ctypes.c_void_p), ("packed", ctypes.c_void_p), ("wdeq", ctypes.c_void_p),
                ("lb", ctypes.c_void_p), ("state", ctypes.c_void_p), ("inv_K", ctypes.c_double), ("eps", ctypes.c_float),
                ("eps1", ctypes.c_float), ("K", ctypes.c_int), ("N", ctypes.c_int), ("seg_rows", ctypes.c_int),
                ("pad", ctypes.c_int)]


class DecodeEngine(NotCopied):
    CHUNK = 32          # steps whose input tokens the recorded graph keeps before the host has to fetch them
    SPIN = 1 << 15      # polling rounds a resident workgroup waits for its input before it gives up (mmf_decode_layers)

    @classmethod
    def for_model(cls, model, batch_size: int, use_graph: bool = True, fuse: bool = True, resident: Optional[bool] = None):
        engines = model.__dict__.setdefault("_decode_engines", {})
        key = (batch_size, use_graph, fuse, resident)
        eng = engines.get(key)
        if eng is None or eng.stale():
            eng = cls(model, batch_size, use_graph, fuse, resident)
            engines[key] = eng
        return eng

    def __init__(self, model, batch_size: int, use_graph: bool = True, fuse: bool = True, resident: Optional[bool] = None):
        cfg = model.config
        if getattr(cfg, "use_short_conv", False):
            raise NotImplementedError("DecodeEngine has no convolution state: models with use_short_conv decode through "
                                      "the module path (generate() does so by itself)")
        self.lib = L.load()
        self.B = B = batch_size
        emb = model.model.embeddings.weight
        self.dev = dev = L.require_gpu(emb)
        self.dtype = dt = emb.dtype
        self.dt_id = L.dtype_id(dt)
        self.H = H = cfg.hidden_size
        self.V = cfg.vocab_size
        self.L = len(model.model.layers)
        self.eps = float(cfg.rms_norm_eps)
        self.use_graph = use_graph
        # what the operands below were taken from: modules, parameters (object, version, address); nothing here leads back to the model,
        # which holds this engine
        dicts = [m.__dict__ for m in model.modules()]
        self._children = [(d["_modules"], k, c) for d in dicts for k, c in d["_modules"].items()]
        self._parameters = [(d["_parameters"], k, p, p._version, p.data_ptr()) for d in dicts
                            for k, p in d["_parameters"].items() if p is not None]
        self._absent = [(d["_parameters"], k) for d in dicts for k, p in d["_parameters"].items() if p is None]
        self._blocks = model.model.layers._modules

        attn0 = model.model.layers[0].attn
        self.D = D = attn0.input_dim
        self.I = I = model.model.layers[0].mlp.intermediate_size
        lbs = model.model.lower_bound_rows() if cfg.use_lower_bound else None

        def z(*shape, dtype=dt):
            return torch.zeros(*shape, dtype=dtype, device=dev)

        w = lambda norm, n: F_.vector(norm.weight, n, "norm weight")

        def codes(proj, n, k):
            """A projection's packed weight: the launches take every layer's sizes from the first one's, the vocabulary's from the configuration."""
            pw = proj.packed_weight()
            if (pw.n, pw.k) != (n, k):
                raise NotImplementedError(f"DecodeEngine: a projection {pw.k} -> {pw.n} where the model's are {k} -> {n}; "
                                          "generate(use_graph=False) decodes layers of different widths")
            return pw

        if tuple(emb.shape) != (self.V, H):
            raise NotImplementedError(f"DecodeEngine: an embedding {tuple(emb.shape)} in a model of {self.V} x {H}; generate(use_graph=False) takes it")

        # ---- per-layer operands (references keep the packed weights alive)
        self.layers = []
        for li, blk in enumerate(model.model.layers):
            a, m = blk.attn, blk.mlp
            ent = {
                "attn_norm": w(blk.attn_norm, H), "mlp_norm": w(blk.mlp_norm, H), "g_norm": w(a.g_norm, D), "g_eps": float(a.g_norm.eps),
                "ifg": a._stacked_weight() if self._stackable(a) else None,
                # None where the three inner norms agree (one row of codes serves i, f and g), else the three weights
                "norms": None if a._stacked_ifg() is not None else [w(p.norm, H) for p in (a.i_proj, a.f_proj, a.g_proj)],
                "projs": [(codes(p, D, H), w(p.norm, H), self._eps_of(p)) for p in (a.i_proj, a.f_proj, a.g_proj)],
                "o": (codes(a.o_proj, H, D), w(a.o_proj.norm, D), self._eps_of(a.o_proj)),
                "gate": (codes(m.gate_proj, 2 * I, H), w(m.gate_proj.norm, H), self._eps_of(m.gate_proj)),
                "down": (codes(m.down_proj, H, I), w(m.down_proj.norm, I), self._eps_of(m.down_proj)),
                "lb": F_.lower_bound_row(lbs[li], D) if lbs is not None and li > 0 else None,
                "state": z(B, D, dtype=torch.float32),
            }
            for p in (a.i_proj, a.f_proj, a.g_proj, a.o_proj, m.gate_proj, m.down_proj):
                if p.bias is not None:
                    raise NotImplementedError("DecodeEngine: BitLinear bias is not on the model path")
            self.layers.append(ent)
        self.final_norm = w(model.model.norm, H)
        self.head = (codes(model.lm_head, self.V, H), w(model.lm_head.norm, H), self._eps_of(model.lm_head))
        self.table = emb.detach().contiguous()

        # ---- static activation buffers
        self.tok = torch.zeros(B, dtype=torch.int64, device=dev)
        # every step records the token it was fed: row t of the history is step t's, modulo CHUNK, counted per batch row
        self.history = torch.zeros(self.CHUNK, B, dtype=torch.int64, device=dev)
        self.pos = torch.zeros(B, dtype=torch.int32, device=dev)
        # what a drawing step reads: temperature, top_p and top_k, and the uniform numbers of the steps that leave pos at t in row t
        self.draw_params = torch.zeros(3, dtype=torch.float32, device=dev)
        self.draw_u = torch.zeros(self.CHUNK, B, dtype=torch.float32, device=dev)
        self.h = z(B, H)            # residual stream
        self.hn = z(B, H)
        self.ifg = z(B, 3 * D)
        self.o = z(B, D)
        self.o2 = z(B, D)
        self.a = z(B, H)
        self.res = z(B, H)
        self.y = z(B, 2 * I)
        self.zb = z(B, I)
        self.logits = z(B, self.V)
        kmax = max(H, D, I)
        # codes, scales and code sums of one row block, or of the three that i, f and g with norms of their own take
        nbytes = max(self.lib.mmf_codes_bytes(B, kmax, 1), 3 * self.lib.mmf_codes_bytes(B, H, 1))
        self.q = torch.zeros(nbytes, dtype=torch.int8, device=dev)
        self.deq = z(3 * B, dtype=torch.float32)
        self.qsum = torch.zeros(3 * B, dtype=torch.int32, device=dev)
        self.gemv = B <= F_.GEMV_MAX_M
        self.fused = fuse and self._can_fuse()
        self.fused_mfma = fuse and self._can_fuse_mfma()
        # a layer whose i, f and g have inner norms of their own: every layer of the resident launch then has three (equal ones repeated)
        self.norms = 3 if any(ent["norms"] is not None for ent in self.layers) else 1
        # resident=None: the one-launch layer chain whenever the model fits it; True insists; False never
        self.resident = self.fused and resident is not False and self._can_run_resident()
        if resident and not self.resident:
            raise L.MMFError("DecodeEngine: this model / batch / device does not fit the resident layer chain")
        if self.resident:
            self._build_resident()
        self.graphs = {}            # recorded steps, by whether they draw their token
        self.probed = False         # the resident chain's workgroups have been seen to be resident at once

    @classmethod
    def _stackable(cls, attn):
        projs = (attn.i_proj, attn.f_proj, attn.g_proj)
        return (attn.input_dim % 32 == 0 and all(p.bias is None and p.norm.weight is not None for p in projs)
                and len({cls._eps_of(p) for p in projs}) == 1)

    @staticmethod
    def _eps_of(p):
        return float(p.norm.eps if getattr(p, "fused_eps", None) is None else p.fused_eps)

    def stale(self):
        """Whether a module or parameter the engine was built on has been replaced or written since, or a layer or an absent parameter
        has come."""
        for d, k, p, version, address in self._parameters:
            if d.get(k) is not p or p._version != version or p.data_ptr() != address:
                return True
        for d, k, c in self._children:
            if d.get(k) is not c:
                return True
        return len(self._blocks) != self.L or any(d.get(k) is not None for d, k in self._absent)

    # ------------------------------------------------------------------ launches
    def _bitlinear(self, x, pw_nw_eps, out, n_k, addend=None):
        pw, nw, eps = pw_nw_eps
        lib, s, B = self.lib, L.stream(), self.B
        n, k = n_k
        nw_id = L.dtype_id(nw.dtype)
        if self.gemv and k <= lib.mmf_bitlinear_gemv_max_k():
            L.check(lib.mmf_bitlinear_gemv(x.data_ptr(), nw.data_ptr(), pw.packed.data_ptr(), pw.wdeq.data_ptr(),
                                           pw.seg_rows, None, L.ptr(addend), out.data_ptr(), B, k, n, eps, self.dt_id,
                                           nw_id, s), "mmf_bitlinear_gemv")
        else:
            L.check(lib.mmf_rmsnorm_quant(x.data_ptr(), None, nw.data_ptr(), self.q.data_ptr(), self.deq.data_ptr(),
                                          self.qsum.data_ptr(), None, B, k, eps, self.dt_id, self.dt_id, nw_id, 1, s),
                    "mmf_rmsnorm_quant")
            L.check(lib.mmf_bitlinear_mfma(self.q.data_ptr(), self.deq.data_ptr(), self.qsum.data_ptr(),
                                           pw.packed.data_ptr(), pw.wdeq.data_ptr(), pw.seg_rows, None, L.ptr(addend),
                                           out.data_ptr(), n, B, k, n, self.dt_id, -1, s), "mmf_bitlinear_mfma")

    # prologue / epilogue ids of mmf_bitlinear_gemv_fused
    PLAIN, NORM, RESNORM, GATEDNORM, SWIGLU = 0, 1, 2, 3, 4
    E_PLAIN, E_STEP, E_SWIGLU = 0, 1, 2

    def _fused(self, pro, epi, x, ldx, aux, ldaux, res_out, w1, eps1, pw_nw_eps, out, g_out, lb, state, n, k,
               addend=None):
        pw, nw, eps = pw_nw_eps
        L.check(self.lib.mmf_bitlinear_gemv_fused(
            pro, epi, x.data_ptr(), ldx, L.ptr(aux), ldaux, L.ptr(res_out), L.ptr(w1), eps1, nw.data_ptr(), eps,
            pw.packed.data_ptr(), pw.wdeq.data_ptr(), pw.seg_rows, None, L.ptr(addend), out.data_ptr(), L.ptr(g_out),
            L.ptr(lb), L.ptr(state), self.B, k, n, self.dt_id, L.dtype_id(nw.dtype), L.stream()), "mmf_bitlinear_gemv_fused")

    # ------------------------------------------------------------------ resident layer chain (batch 1)
    def _can_run_resident(self):
        props = torch.cuda.get_device_properties(self.dev)
        return (self.B == 1 and self.dtype in (torch.bfloat16, torch.float16) and self.final_norm.dtype == self.dtype
                and bool(self.lib.mmf_decode_layers_fits(self.norms, self.L, self.H, self.D, self.I))
                and props.multi_processor_count >= 256)

    def _build_resident(self):
        H, D, I = self.H, self.D, self.I
        assert self.lib.mmf_decode_layers_phase_bytes() == ctypes.sizeof(_Phase)
        table = (_Phase * (4 * self.L + 1))()            # the last record is the final norm + lm_head

        def fill(rec, w1, eps1, pw_nw_eps, k, n, lb=None, state=None):
            pw, nw, eps = pw_nw_eps
            rec.w1 = w1.data_ptr() if w1 is not None else None
            rec.norm_w, rec.packed, rec.wdeq = nw.data_ptr(), pw.packed.data_ptr(), pw.wdeq.data_ptr()
            assert nw.is_contiguous() and (w1 is None or w1.is_contiguous())
            rec.lb = lb.data_ptr() if lb is not None else None
            rec.state = state.data_ptr() if state is not None else None
            rec.inv_K, rec.eps, rec.eps1, rec.K, rec.N, rec.seg_rows = 1.0 / k, eps, eps1, k, n, pw.seg_rows

        for li, ent in enumerate(self.layers):
            nw = ent["projs"][0][1]
            if self.norms == 3:
                nw = ent["norm3"] = torch.stack(ent["norms"] or [nw] * 3)
            fill(table[4 * li], ent["attn_norm"], self.eps, (ent["ifg"], nw, ent["projs"][0][2]), H, 3 * D, ent["lb"], ent["state"])
            fill(table[4 * li + 1], ent["g_norm"], ent["g_eps"], ent["o"], D, H)
            fill(table[4 * li + 2], ent["mlp_norm"], self.eps, ent["gate"], H, 2 * I)
            fill(table[4 * li + 3], None, 0.0, ent["down"], I, H)
        fill(table[4 * self.L], self.final_norm, self.eps, self.head, H, self.V)
        raw = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8)
        self.phases = raw.to(self.dev)
        # tagged hand-off words: every row in `copies` copies (one per XCD), [copies, n] each, in the kernel's order
        R = self.lib.mmf_decode_layers_copies()
        sizes = [H, H, D, D, H, I]                          # h0, h1, o, g, attn, z
        words = torch.zeros(self.lib.mmf_decode_layers_words(H, D, I), dtype=torch.int32, device=self.dev)
        self.words, off = [], 0
        for n in sizes:
            self.words.append(words[off:off + R * n].view(R, n))
            off += R * n
        assert off == words.numel()
        self._words = words
        self.am_words = torch.zeros(256, dtype=torch.int64, device=self.dev)
        self.epoch = torch.zeros(1, dtype=torch.int32, device=self.dev)
        self.err = torch.zeros(1, dtype=torch.int32, device=self.dev)

    def _launch_layers(self, with_head: bool, trace: Optional[torch.Tensor] = None, delay: int = 6):
        head = self.phases.data_ptr() + 4 * self.L * ctypes.sizeof(_Phase) if with_head else None
        args = (self.phases.data_ptr(), self.L, self.table.data_ptr(), self.tok.data_ptr(), self.V, self._words.data_ptr(),
                self.h.data_ptr(), head, self.logits.data_ptr(), self.am_words.data_ptr(), self.tok.data_ptr(),
                self.epoch.data_ptr(), self.err.data_ptr())
        record = (self.history.data_ptr(), self.pos.data_ptr(), self.CHUNK)
        if trace is None:
            L.check(self.lib.mmf_decode_layers_norms(self.norms, *args, *record, self.H, self.D, self.I, self.SPIN, self.dt_id, L.stream()),
                    "mmf_decode_layers_norms")
        else:
            assert self.norms == 1, "the traced kernel is built for shared inner norms"
            L.check(self.lib.mmf_decode_layers_traced(*args, trace.data_ptr(), self.H, self.D, self.I, self.SPIN, delay, self.dt_id,
                                                      L.stream()), "mmf_decode_layers_traced")

    def link_trace(self, delay: int = 6) -> torch.Tensor:
        """One resident step with the kernel's cycle trace on: int64 [256 workgroups, 128 links, 12 stamps] (see
        mmf_decode_layers_traced in include/mmf_diag.h), on the host."""
        assert self.resident
        t = torch.zeros(self.lib.mmf_decode_layers_trace_words(), dtype=torch.int64, device=self.dev)
        self._launch_layers(True, trace=t, delay=delay)
        torch.cuda.synchronize(self.dev)
        return t.view(256, 128, 12).cpu()

    def _launch_step_resident(self, draw):
        self._launch_layers(True)       # the whole step: final norm, lm_head and argmax are the launch's last two links
        if draw:
            self._choose(True)

    def resident_ok(self) -> bool:
        """False once a wait inside the resident layer chain ran out of polling rounds (host synchronisation)."""
        return not self.resident or int(self.err.item()) == 0

    def _reset_resident(self):
        """Bring the hand-off words back to their initial state.  A launch whose wait timed out may have had a late
        workgroup read the tag base after workgroup 0 advanced it (the base is only published safely when every poll
        succeeded), and so have left words that carry tags of the NEXT launch; a later launch would accept them as its
        own.  With every word, the tag base and the error word zero the next launch starts like the first one.  The
        caller has synchronised with the device (it has read the error word)."""
        self._words.zero_()
        self.am_words.zero_()
        self.epoch.zero_()
        self.err.zero_()

    def check(self):
        """Raise if a wait inside the resident layer chain timed out since the engine was built: its workgroups were
        not all resident at once (other work held CUs), so the steps since then are invalid.  One host synchronisation;
        callers run it once per generation, not per step.  The engine is reset and can be used again."""
        if not self.resident_ok():
            self._reset_resident()
            raise L.MMFError("DecodeEngine: a wait inside the resident layer chain timed out (were other kernels running "
                             "on this device?); the tokens of this generation are invalid. Build the engine with "
                             "resident=False to decode with one launch per BitLinear.")

    def _embed(self):
        L.check(self.lib.mmf_embedding_record(self.table.data_ptr(), self.tok.data_ptr(), self.h.data_ptr(), self.B, self.H, self.V,
                                              self.history.data_ptr(), self.pos.data_ptr(), self.CHUNK, self.dt_id, L.stream()),
                "mmf_embedding_record")

    def _choose(self, draw):
        """The step's token from its logits: the largest, or the draw that run() has set up."""
        if draw:
            L.check(self.lib.mmf_sample_top_p_recorded(self.logits.data_ptr(), self.V, self.B, self.V, self.draw_params.data_ptr(),
                                                       self.draw_u.data_ptr(), self.pos.data_ptr(), self.tok.data_ptr(), self.dt_id,
                                                       L.stream()), "mmf_sample_top_p_recorded")
        else:
            L.check(self.lib.mmf_argmax(self.logits.data_ptr(), self.V, self.B, self.V, self.tok.data_ptr(), self.dt_id, L.stream()),
                    "mmf_argmax")

    def _launch_step_fused(self, ends=True, draw=False):
        """Batch <= GEMV_MAX_M: four launches per layer, every elementwise op folded into a GEMV.
        ends=False leaves out the embedding gather and the choice of the token (the 4L+1 GEMV launches only)."""
        lib, s, B, H, D, I = self.lib, L.stream(), self.B, self.H, self.D, self.I
        if ends:
            self._embed()
        g_buf = self.ifg.view(-1)[:B * D].view(B, D)
        for ent in self.layers:
            if ent["norms"] is not None:
                pw, n = ent["ifg"], ent["norms"]
                L.check(lib.mmf_bitlinear_gemv_multi(
                    self.E_STEP, self.h.data_ptr(), H, ent["attn_norm"].data_ptr(), self.eps, n[0].data_ptr(), n[1].data_ptr(),
                    n[2].data_ptr(), ent["projs"][0][2], pw.packed.data_ptr(), pw.wdeq.data_ptr(), pw.seg_rows, self.o.data_ptr(),
                    g_buf.data_ptr(), L.ptr(ent["lb"]), ent["state"].data_ptr(), B, H, 3 * D, self.dt_id, L.dtype_id(n[0].dtype), s),
                    "mmf_bitlinear_gemv_multi")
            else:
                self._fused(self.NORM, self.E_STEP, self.h, H, None, 0, None, ent["attn_norm"], self.eps,
                            (ent["ifg"], ent["projs"][0][1], ent["projs"][0][2]), self.o, g_buf, ent["lb"], ent["state"],
                            3 * D, H)
            self._fused(self.GATEDNORM, self.E_PLAIN, g_buf, D, self.o, D, None, ent["g_norm"], ent["g_eps"], ent["o"],
                        self.a, None, None, None, H, D)
            self._fused(self.RESNORM, self.E_SWIGLU, self.a, H, self.h, H, self.res, ent["mlp_norm"], self.eps,
                        ent["gate"], self.zb, None, None, None, 2 * I, H)
            self._fused(self.PLAIN, self.E_PLAIN, self.zb, I, None, 0, None, None, 0.0, ent["down"], self.h, None, None,
                        None, H, I, addend=self.res)
        self._fused(self.NORM, self.E_PLAIN, self.h, H, None, 0, None, self.final_norm, self.eps, self.head, self.logits,
                    None, None, None, self.V, H)
        if ends:
            self._choose(draw)

    def fused_step_bytes(self, with_head: bool = True):
        """Algorithmic bytes of the 4L (+1 with head) fused BitLinears of one batch-B step: 2-bit weights once, plus
        each link's activation / norm-weight / state reads and its outputs."""
        B, H, D, I, V, e = self.B, self.H, self.D, self.I, self.V, self.h.element_size()
        per_layer = ((3 * D * H + H * D + 2 * I * H + H * I) // 4        # packed weights of i/f/g, o, gate, down
                     + B * (H * e + 2 * D * e + 8 * D) + 2 * H * e + 4 * D  # A: x; o, g out; state rd+wr; two norm weights, lb
                     + B * (2 * D * e + H * e) + 2 * D * e                  # B: g, o in; a out; two norm weights
                     + B * (2 * H * e + H * e + I * e) + 2 * H * e          # C: a, h in; res, z out; two norm weights
                     + B * (I * e + 2 * H * e) + I * e)                     # D: z, res in; h out; norm weight
        head = V * H // 4 + B * (H * e + V * e) + 2 * H * e
        return self.L * per_layer + (head if with_head else 0)

    def _qfused(self, pro, x, ldx, aux, ldaux, aux2, ldaux2, res_out, w1, eps1, nw, eps, lb, state, k):
        L.check(self.lib.mmf_rmsnorm_quant_fused(
            pro, x, ldx, aux, ldaux, aux2, ldaux2, L.ptr(res_out), L.ptr(w1), eps1, nw.data_ptr(), eps, L.ptr(lb),
            L.ptr(state), self.q.data_ptr(), self.deq.data_ptr(), self.qsum.data_ptr(), self.B, k, self.dt_id,
            L.dtype_id(nw.dtype), L.stream()), "mmf_rmsnorm_quant_fused")

    def _mfma(self, pw, out, n, k, addend=None):
        L.check(self.lib.mmf_bitlinear_mfma(self.q.data_ptr(), self.deq.data_ptr(), self.qsum.data_ptr(),
                                            pw.packed.data_ptr(), pw.wdeq.data_ptr(), pw.seg_rows, None, L.ptr(addend),
                                            out.data_ptr(), n, self.B, k, n, self.dt_id, -1, L.stream()), "mmf_bitlinear_mfma")

    def _launch_step_mfma_fused(self, draw):
        """Batch > GEMV_MAX_M: eight launches per layer -- each BitLinear is a fused prologue+quantiser row kernel
        (norm / recurrence step + gated norm / residual norm / swiglu folded in) and a matrix-core contraction."""
        lib, s, B, H, D, I = self.lib, L.stream(), self.B, self.H, self.D, self.I
        esz = self.h.element_size()
        self._embed()
        ifg = self.ifg.data_ptr()
        for ent in self.layers:
            nw, eps = ent["projs"][0][1], ent["projs"][0][2]
            if ent["norms"] is not None:
                pw, n = ent["ifg"], ent["norms"]
                L.check(lib.mmf_rmsnorm_quant_multi(
                    self.h.data_ptr(), H, ent["attn_norm"].data_ptr(), self.eps, n[0].data_ptr(), n[1].data_ptr(), n[2].data_ptr(), eps,
                    self.q.data_ptr(), self.deq.data_ptr(), self.qsum.data_ptr(), B, H, self.dt_id, L.dtype_id(nw.dtype), s),
                    "mmf_rmsnorm_quant_multi")
                L.check(lib.mmf_bitlinear_mfma_multi(
                    self.q.data_ptr(), lib.mmf_codes_bytes(B, H, 1), self.deq.data_ptr(), self.qsum.data_ptr(), pw.packed.data_ptr(),
                    pw.wdeq.data_ptr(), pw.seg_rows, self.ifg.data_ptr(), 3 * D, B, H, 3 * D, self.dt_id, -1, s),
                    "mmf_bitlinear_mfma_multi")
            else:
                self._qfused(1, self.h.data_ptr(), H, None, 0, None, 0, None, ent["attn_norm"], self.eps, nw, eps, None, None, H)
                self._mfma(ent["ifg"], self.ifg, 3 * D, H)
            self._qfused(3, ifg, 3 * D, ifg + D * esz, 3 * D, ifg + 2 * D * esz, 3 * D, None, ent["g_norm"], ent["g_eps"],
                         ent["o"][1], ent["o"][2], ent["lb"], ent["state"], D)
            self._mfma(ent["o"][0], self.a, H, D)
            self._qfused(2, self.a.data_ptr(), H, self.h.data_ptr(), H, None, 0, self.res, ent["mlp_norm"], self.eps,
                         ent["gate"][1], ent["gate"][2], None, None, H)
            gate = ent["gate"][0]
            L.check(lib.mmf_bitlinear_mfma_swiglu(self.q.data_ptr(), self.deq.data_ptr(), self.qsum.data_ptr(), gate.packed.data_ptr(),
                                                  gate.wdeq.data_ptr(), gate.seg_rows, self.zb.data_ptr(), I, B, H, 2 * I, self.dt_id, s),
                    "mmf_bitlinear_mfma_swiglu")
            self._qfused(0, self.zb.data_ptr(), I, None, 0, None, 0, None, None, 0.0, ent["down"][1], ent["down"][2], None, None, I)
            self._mfma(ent["down"][0], self.h, H, I, addend=self.res)
        self._qfused(1, self.h.data_ptr(), H, None, 0, None, 0, None, self.final_norm, self.eps, self.head[1], self.head[2],
                     None, None, H)
        self._mfma(self.head[0], self.logits, self.V, H)
        self._choose(draw)

    def _can_fuse_mfma(self):
        same_dt = all(t.dtype == self.final_norm.dtype for e in self.layers
                      for t in (e["attn_norm"], e["mlp_norm"], e["g_norm"], e["o"][1], e["gate"][1], e["down"][1],
                                *(p[1] for p in e["projs"]))) and self.head[1].dtype == self.final_norm.dtype
        return (not self.gemv and same_dt and all(e["ifg"] is not None for e in self.layers)
                and max(self.H, self.D, self.I) <= 8192 and (3 * self.D) % 8 == 0 and self.I % 32 == 0)

    def _can_fuse(self):
        kmax = self.lib.mmf_bitlinear_gemv_max_k()
        same_dt = all(t.dtype == self.final_norm.dtype for e in self.layers
                      for t in (e["attn_norm"], e["mlp_norm"], e["g_norm"], e["o"][1], e["gate"][1], e["down"][1],
                                *(p[1] for p in e["projs"]))) and self.head[1].dtype == self.final_norm.dtype
        return (self.gemv and same_dt and all(e["ifg"] is not None for e in self.layers)
                and max(self.H, self.D, self.I) <= kmax and self.D % 32 == 0 and self.I % 32 == 0)

    def _launch_step(self, draw=False):
        if self.resident:
            return self._launch_step_resident(draw)
        if self.fused:
            return self._launch_step_fused(draw=draw)
        if self.fused_mfma:
            return self._launch_step_mfma_fused(draw)
        lib, s, B, H, D, I = self.lib, L.stream(), self.B, self.H, self.D, self.I
        dt, esz = self.dt_id, self.h.element_size()
        wid = L.dtype_id(self.final_norm.dtype)
        self._embed()
        for ent in self.layers:
            L.check(lib.mmf_rmsnorm(self.h.data_ptr(), None, ent["attn_norm"].data_ptr(), self.hn.data_ptr(), None, B, H,
                                    self.eps, dt, dt, wid, s), "mmf_rmsnorm")
            if ent["norms"] is None:
                self._bitlinear(self.hn, (ent["ifg"], ent["projs"][0][1], ent["projs"][0][2]), self.ifg, (3 * D, H))
                ip, fp, gp, ld = self.ifg.data_ptr(), self.ifg.data_ptr() + D * esz, self.ifg.data_ptr() + 2 * D * esz, 3 * D
            else:
                # three separate projections into the three column blocks of a [3, B, D] layout
                bufs = self.ifg.view(3, B, D)
                for j in range(3):
                    self._bitlinear(self.hn, ent["projs"][j], bufs[j], (D, H))
                ip, fp, gp, ld = bufs[0].data_ptr(), bufs[1].data_ptr(), bufs[2].data_ptr(), D
            L.check(lib.mmf_hgrn_step(ip, ld, fp, ld, L.ptr(ent["lb"]), None, ent["state"].data_ptr(), self.o.data_ptr(),
                                      B, D, dt, s), "mmf_hgrn_step")
            L.check(lib.mmf_rmsnorm_swishgate(gp, ld, self.o.data_ptr(), None, ent["g_norm"].data_ptr(),
                                              self.o2.data_ptr(), None, B, D, ent["g_eps"], dt, dt, wid, s),
                    "mmf_rmsnorm_swishgate")
            self._bitlinear(self.o2, ent["o"], self.a, (H, D))
            L.check(lib.mmf_rmsnorm(self.a.data_ptr(), self.h.data_ptr(), ent["mlp_norm"].data_ptr(), self.hn.data_ptr(),
                                    self.res.data_ptr(), B, H, self.eps, dt, dt, wid, s), "mmf_rmsnorm")
            self._bitlinear(self.hn, ent["gate"], self.y, (2 * I, H))
            L.check(lib.mmf_swiglu(self.y.data_ptr(), 2 * I, self.y.data_ptr() + I * esz, 2 * I, self.zb.data_ptr(), B, I,
                                   dt, s), "mmf_swiglu")
            self._bitlinear(self.zb, ent["down"], self.h, (H, I), addend=self.res)
        L.check(lib.mmf_rmsnorm(self.h.data_ptr(), None, self.final_norm.data_ptr(), self.hn.data_ptr(), None, B, H,
                                self.eps, dt, dt, wid, s), "mmf_rmsnorm")
        self._bitlinear(self.hn, self.head, self.logits, (self.V, H))
        self._choose(draw)

    def _prepare(self, draw):
        """Warm-up launches on a side stream (module loading, attribute setting); then the step is recorded, unless it is a single
        launch (as a graph of one node the resident step takes 399 us for 394)."""
        saved = [e["state"].clone() for e in self.layers]
        tok, pos = self.tok.clone(), self.pos.clone()
        side = torch.cuda.Stream(device=self.dev)
        side.wait_stream(torch.cuda.current_stream(self.dev))
        with torch.cuda.stream(side):
            self._launch_step(draw)
        torch.cuda.current_stream(self.dev).wait_stream(side)
        torch.cuda.synchronize(self.dev)
        if self.resident and not self.resident_ok():
            # the workgroups were not all resident at once (another stream or process holds CUs): use the launch chain
            warnings.warn("DecodeEngine: the resident layer chain timed out waiting for its workgroups; "
                          "falling back to one launch per BitLinear")
            self.resident = False
            self._reset_resident()
            for e, sv in zip(self.layers, saved):
                e["state"].copy_(sv)
            self.tok.copy_(tok)
            with torch.cuda.stream(side):
                self._launch_step(draw)
            torch.cuda.current_stream(self.dev).wait_stream(side)
            torch.cuda.synchronize(self.dev)
        self.probed = True
        if not self.resident:
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                self._launch_step(draw)
            torch.cuda.synchronize(self.dev)
            self.graphs[draw] = g
        for e, sv in zip(self.layers, saved):     # undo the warm-up step's state update
            e["state"].copy_(sv)
        self.tok.copy_(tok)
        self.pos.copy_(pos)

    # ------------------------------------------------------------------ public
    def load_state(self, states: Optional[List[torch.Tensor]]):
        """Set the per-layer recurrent states ([B, *, D] tensors, or None for zeros)."""
        if states is None:
            torch._foreach_zero_([e["state"] for e in self.layers])
        else:
            # one launch for all layers (a copy per layer costs more than a decode step's layer)
            torch._foreach_copy_([e["state"] for e in self.layers],
                                 [s.reshape(self.B, self.D).to(device=self.dev, dtype=torch.float32) for s in states])

    def export_state(self):
        return [e["state"].clone() for e in self.layers]

    def advance(self, draw: bool = False):
        """One decode step from the token buffer; leaves logits in self.logits and the greedy (``draw``: the drawn, see run)
        next token in the token buffer (no host synchronisation)."""
        with L.on(self.dev):
            if self.use_graph and not (self.probed if self.resident else draw in self.graphs):
                self._prepare(draw)
            if self.use_graph and not self.resident:
                self.graphs[draw].replay()
            else:
                self._launch_step(draw)

    def step(self, tokens: torch.Tensor) -> torch.Tensor:
        """Feed `tokens` [B]; returns the logits buffer [B, V] (overwritten by the next step)."""
        self.tok.copy_(tokens.reshape(self.B))
        self.advance()
        return self.logits

    def run(self, n_steps: int, pick=None, seen=None, draw=None) -> torch.Tensor:
        """n_steps self-feeding steps from the token buffer; returns the [n_steps + 1, B] tokens: what the buffer held, then what
        it held after each step.  pick(t), when given, replaces the token step t chose; draw =
        (uniform numbers [n_steps, B], top_p, temperature, top_k) has the steps draw theirs as functional.sample_top_p does.  seen(tokens [t + 1, B]), when given, is
        asked every CHUNK steps whether to stop there.  No host synchronisation of its own."""
        out = torch.empty(n_steps + 1, self.B, dtype=torch.int64, device=self.dev)
        self.pos.zero_()
        if draw is not None:
            u, top_p, temperature, top_k = draw
            params = struct.pack("=ffi", temperature, min(max(top_p, 0.0), 1.0), top_k if top_k < self.V else 0)
            self.draw_params.view(torch.uint8).copy_(torch.frombuffer(bytearray(params), dtype=torch.uint8))
        done = 0
        while done < n_steps:
            n = min(self.CHUNK, n_steps - done)
            if draw is not None:                                # step t of the chunk leaves pos at (t + 1) % CHUNK
                m = min(n, self.CHUNK - 1)
                self.draw_u[1:m + 1].copy_(u[done:done + m])
                if m < n:
                    self.draw_u[0].copy_(u[done + m])
            for t in range(done, done + n):
                self.advance(draw is not None)
                if pick is not None:
                    pick(t)
            out[done:done + n].copy_(self.history[:n])
            done += n
            if seen is not None or done == n_steps:
                out[done].copy_(self.tok)
            if seen is not None and seen(out[:done + 1]):
                break
        if n_steps == 0:
            out[0].copy_(self.tok)
        return out[:done + 1]

    def greedy(self, first_tokens: torch.Tensor, n_steps: int) -> torch.Tensor:
        """Run n_steps self-feeding greedy steps starting from first_tokens [B]; returns the
        [B, n_steps] tokens chosen after each step.  One host synchronisation at the end."""
        self.tok.copy_(first_tokens.reshape(self.B))
        out = self.run(n_steps)[1:]
        self.check()
        return out.t().contiguous()
