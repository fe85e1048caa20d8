"""A training step with whole blocks as autograd ops against the op-by-op composition (which a hook anywhere in the model
brings back): same loss bit for bit, gradients within rounding.  Widths on both sides of the row kernels' passes, row
counts below and above their grid, masks, frozen weights, no lower bounds.  A block's gradients against a composition in
double precision: no further off than the op-by-op one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def step(model, ids, mask, hook):
    hooks = [m.register_forward_hook(lambda *a: None) for layer in model.model.layers for m in (layer.attn.g_norm,)] if hook else []
    if hook:
        hooks.append(model.model.norm.register_forward_hook(lambda *a: None))
    model.zero_grad(set_to_none=True)
    loss = model(input_ids=ids, attention_mask=mask, labels=ids).loss
    loss.backward()
    for h in hooks:
        h.remove()
    return loss.detach(), {n: p.grad for n, p in model.named_parameters()}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden,b,t,masked,lb", [(96, 1, 5, False, True), (160, 3, 33, True, True), (512, 2, 600, False, False),
                                                  (2048, 1, 70, False, True), (2560, 1, 40, True, True)])
def test_block_step_equals_the_composition(dev, dtype, hidden, b, t, masked, lb):
    import matmulfreellm_amd as mm
    torch.manual_seed(23)
    model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=200, hidden_size=hidden, num_hidden_layers=2, use_lower_bound=lb))
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name:
                p.copy_(0.5 + torch.rand(p.shape))
            if name.endswith("lower_bounds"):
                p.copy_(torch.randn(p.shape))
    model = model.to(dev, dtype).train()
    model.model.layers[0].mlp.down_proj.weight.requires_grad_(False)
    ids = torch.randint(0, 200, (b, t), device=dev)
    mask = (torch.arange(t, device=dev) >= torch.arange(b, device=dev).view(-1, 1) + 1).long() if masked else None
    loss, got = step(model, ids, mask, False)
    ref_loss, want = step(model, ids, mask, True)
    assert torch.equal(loss, ref_loss)
    for name in want:
        if want[name] is None:
            assert got[name] is None, name
            continue
        g, w = got[name].double(), want[name].double()
        err = ((g - w).norm() / w.norm().clamp_min(1e-30)).item()
        assert err < (2e-5 if dtype == torch.float32 else 2e-2), (name, err)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_trained_head_on_a_frozen_body_keeps_the_cache(dev, dtype):
    """Gradients enabled, only the head's parameters ask for one: the body runs as in inference, takes and returns a cache; the
    head's gradients are those of the modules one by one."""
    import matmulfreellm_amd as mm
    torch.manual_seed(29)
    model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=200, hidden_size=96, num_hidden_layers=2)).to(dev, dtype)
    model.model.requires_grad_(False)
    ids, more = (torch.randint(0, 200, (2, n), device=dev) for n in (7, 1))
    with torch.no_grad():
        want = model(input_ids=ids, use_cache=True)
        want_next = model(input_ids=more, past_key_values=want.past_key_values, use_cache=True)
    out = model(input_ids=ids, use_cache=True)
    assert torch.equal(out.logits, want.logits) and out.logits.requires_grad
    step = model(input_ids=more, past_key_values=out.past_key_values, use_cache=True)
    assert torch.equal(step.logits, want_next.logits)
    _, got = step_of(model, ids)
    hook = model.model.norm.register_forward_hook(lambda *a: None)
    _, ref = step_of(model, ids)
    hook.remove()
    assert set(got) == {"lm_head.weight", "lm_head.norm.weight"}
    for name in got:
        err = ((got[name].double() - ref[name].double()).norm() / ref[name].double().norm()).item()
        assert err < (1e-6 if dtype == torch.float32 else 1e-2), (name, err)


def step_of(model, ids):
    model.zero_grad(set_to_none=True)
    loss = model(input_ids=ids, labels=ids).loss
    loss.backward()
    return loss.detach(), {n: p.grad for n, p in model.named_parameters() if p.grad is not None}


def in_64_bits(layer, x, lb, mask, dout):
    """The layer in double precision; every tensor that the kernels materialise takes the value they gave it (straight-through), codes too."""
    import matmulfreellm_amd.functional as F_
    value = lambda v, actual: v + (actual.double() - v).detach()
    attn, mlp = layer.attn, layer.mlp
    leaf = {n: p.detach().double().requires_grad_() for n, p in layer.named_parameters()}
    lbl = lb.detach().double().requires_grad_() if lb is not None else None
    names = {p: n for n, p in layer.named_parameters()}

    def norm(v, w, eps):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + eps) * w

    def bitlinear(v, s, p):
        w = p.norm.weight
        q, deq, _ = F_.rmsnorm_quant(s.reshape(-1, s.shape[-1]), w, eps=p.run_eps())
        codes = q.view(deq.numel(), -1)[:, :s.shape[-1]].double() * deq.double().view(-1, 1)
        y = value(norm(v, leaf[names[w]], p.run_eps()), codes.view(s.shape))
        pw = p.packed_weight()
        w64 = leaf[names[p.weight]]
        wq = w64 + (F_.unpack_ternary(pw).double() * pw.wdeq.double() - w64).detach()
        out = F_.bitlinear(s, w, pw, eps=p.run_eps())
        return value(y @ wq.t(), out), out

    x64 = x.detach().double().requires_grad_()
    s = F_.rmsnorm(x, layer.attn_norm.weight, eps=layer.attn_norm.eps)
    v = value(norm(x64, leaf["attn_norm.weight"], layer.attn_norm.eps), s)
    (vi, i), (vf, f), (vg, g) = (bitlinear(v, s, p) for p in (attn.i_proj, attn.f_proj, attn.g_proj))
    xin, gate = F_.hgrn_gate(i, f, lb, mask)
    sig = torch.sigmoid(vf)
    vgate = sig if lbl is None else lbl + (1 - lbl) * sig
    vx = vi * torch.sigmoid(vi) * (1 - vgate)
    if mask is not None:
        vx = vx * mask.double().unsqueeze(-1)
    vgate, vx = value(vgate, gate), value(vx, xin)
    b, t, D = i.shape
    o, _ = F_.hgrn_recurrent(xin.view(b, 1, t, D), gate.view(b, 1, t, D))
    o = o.view(b, t, D)
    h, hs = torch.zeros(b, D, dtype=torch.float64, device=x.device), []
    for k in range(t):
        h = value(vgate[:, k] * h + vx[:, k], o[:, k])
        hs.append(h)
    vo = torch.stack(hs, 1)
    s = F_.rmsnorm_swishgate(g, o, attn.g_norm.weight, eps=attn.g_norm.eps)
    v = value(norm(vg, leaf["attn.g_norm.weight"], attn.g_norm.eps) * vo * torch.sigmoid(vo), s)
    va, a = bitlinear(v, s, attn.o_proj)
    s, res = F_.rmsnorm(a, layer.mlp_norm.weight, residual=x, eps=layer.mlp_norm.eps, prenorm=True)
    vsum = value(va + x64, a.float() + x.float())             # normalised unrounded, carried on rounded
    vres = value(vsum, res)
    v = value(norm(vsum, leaf["mlp_norm.weight"], layer.mlp_norm.eps), s)
    vy, y = bitlinear(v, s, mlp.gate_proj)
    I = mlp.intermediate_size
    s = F_.swiglu(y[..., :I], y[..., I:])
    v = value(vy[..., :I] * torch.sigmoid(vy[..., :I]) * vy[..., I:], s)
    vz, _ = bitlinear(v, s, mlp.down_proj)
    out = vres + vz
    return torch.autograd.grad(out, [x64] + ([lbl] if lbl is not None else []) + list(leaf.values()), dout.double())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hidden,b,t,masked,lb", [(512, 2, 600, False, False), (1024, 2, 333, False, True), (2560, 2, 40, True, True)])
def test_block_gradients_are_no_further_from_64_bits_than_the_compositions(dev, dtype, hidden, b, t, masked, lb):
    """Both round every tensor between their kernels; the block has fewer of them and contracts the forward's own codes.  Measured, 4 x 256
    rows of 2048 in bf16, block / composition: x 3.4e-3 / 4.0e-3, i, f 5.0e-3 / 5.6e-3, gate 3.3e-3 / 3.7e-3, down 2.3e-3 for both.  Ratios of
    two sums of random roundings: 10 % of leeway (at most 1.05 measured here); a half type's errors stay below 4 unit roundoffs."""
    import matmulfreellm_amd as mm
    from matmulfreellm_amd import block as native
    from matmulfreellm_amd.autograd import BlockFn
    torch.manual_seed(23)
    layer = mm.HGRNBitModel(mm.HGRNBitConfig(vocab_size=200, hidden_size=hidden, num_hidden_layers=2)).layers[1]
    with torch.no_grad():
        for name, p in layer.named_parameters():
            if "norm" in name:
                p.copy_(0.5 + torch.rand(p.shape))
    layer = layer.to(dev, dtype).train()
    x = torch.randn(b, t, hidden, device=dev).to(dtype).requires_grad_()
    low = torch.rand(hidden, device=dev).mul(0.5).requires_grad_() if lb else None
    mask = (torch.arange(t, device=dev) >= torch.arange(b, device=dev).view(-1, 1) + 1).long() if masked else None
    dout = torch.randn(b, t, hidden, device=dev).to(dtype)
    leaves = [x] + ([low] if lb else []) + list(layer.parameters())
    names = ["x"] + (["lower_bound"] if lb else []) + [n for n, _ in layer.named_parameters()]
    plan = native.TrainPlan.of(layer, x)
    out = BlockFn.apply(plan, x, low, mask, *plan.norm_params, *plan.weight_params)
    got = torch.autograd.grad(out, leaves, dout)
    layer.attn.g_norm.register_forward_hook(lambda *a: None)
    composed = layer(x, attention_mask=mask, lower_bound=low)[0]
    assert torch.equal(out, composed)
    ops = torch.autograd.grad(composed, leaves, dout)
    exact = in_64_bits(layer, x.detach(), low.detach() if lb else None, mask, dout)
    for name, a, c, r in zip(names, got, ops, exact):
        block, composition = (((v.double() - r).norm() / r.norm()).item() for v in (a, c))
        assert block <= 1.1 * composition, (name, block, composition)
        assert dtype == torch.float32 or block < 4 * torch.finfo(dtype).eps / 2, (name, block)


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("k", [2048, 2052, 5632])
def test_gradients_take_the_sigmoid_of_the_definition(dev, gated, k):
    """bf16 rows whose gate arguments lie in [-30, -16], where a sigmoid from hardware exp2 alone is up to 30 units of 2^-24 off.  A stored
    gradient misses the exact one by half a spacing of bf16 and at most 14 units: 3 in the sigmoid, 1 in each root, 4 in the gradient
    through the norm, 5 in the products behind it (3.1 measured; with hardware exp2 alone 22 to 27)."""
    import matmulfreellm_amd.functional as F
    from matmulfreellm_amd.autograd import CHAIN_GATED, CHAIN_SWIGLU, _chain_bwd
    torch.manual_seed(k)
    rows = 1024
    gate = (-16 - 14 * torch.rand(rows, k, device=dev)).bfloat16()
    other, dy = torch.randn(rows, k, device=dev).bfloat16(), torch.randn(rows, k, device=dev).bfloat16()
    w1, w2 = ((0.5 + torch.rand(k, device=dev)).bfloat16() for _ in range(2))
    a, v, d64 = gate.double(), other.double(), dy.double()
    sg = torch.sigmoid(a)
    other_grad = torch.empty_like(gate)
    if gated:
        s = F.rmsnorm_swishgate(other, gate, w1, eps=1e-6).double()
        x, aux, kind = other, gate, CHAIN_GATED
        xh = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-6)
    else:
        s = F.swiglu(gate, other).double()
        x, aux, kind = gate, other, CHAIN_SWIGLU
    rstd = torch.rsqrt(s.square().mean(-1, keepdim=True) + 1e-6)
    wd = w2.double() * d64
    d = (wd - s * rstd * (s * rstd * wd).mean(-1, keepdim=True)) * rstd
    got, daux, _, _ = _chain_bwd(kind, x, aux, w1 if gated else None, 1e-6, [w2], 1e-6, [dy], daux=other_grad)
    if gated:
        pairs = [(daux, d * xh * w1.double() * sg * (1 + a * (1 - sg)))]
    else:
        pairs = [(daux, d * a * sg), (got, sg * (1 + a * (1 - sg)) * d * v)]
    for value, want in pairs:
        spacing = torch.exp2(torch.floor(torch.log2(want.abs())) - 7)
        beyond = ((value.double() - want).abs() - spacing / 2) / want.abs()
        beyond = beyond[(wd.abs() > 0.05) & (want != 0)]                 # (the subtraction in d has cancelled nothing there)
        assert beyond.max().item() <= 14 * 2 ** -24


def test_the_backward_of_a_block_takes_no_more_memory_than_with_a_product_at_a_time(dev):
    """8192 rows of 1024 in bf16, beyond the gradients that it returns, in rows of 1024 an input row: at their most, behind the last row kernel, 22.25 are live (dout 1, the
    gradients of gate and up 5.5, of i, f and g 3, of the block's middle 1 and its input 1, of the three projections' inputs 3, six BitLinears'
    de-quantised inputs 7.75) and the stacked weights 0.4; the gradients handed out do not exist yet then, 1.5.  One product at a time, with every
    temporary kept to the end, took 26.6."""
    import matmulfreellm_amd as mm
    from matmulfreellm_amd import block as native
    from matmulfreellm_amd.autograd import BlockFn
    torch.manual_seed(31)
    layer = mm.HGRNBitModel(mm.HGRNBitConfig(vocab_size=200, hidden_size=1024, num_hidden_layers=2)).layers[1].to(dev, torch.bfloat16).train()
    x = torch.randn(8, 1024, 1024, device=dev).bfloat16().requires_grad_()
    low, dout = torch.rand(1024, device=dev).requires_grad_(), torch.randn(8, 1024, 1024, device=dev).bfloat16()
    plan = native.TrainPlan.of(layer, x)
    leaves = [x, low, *layer.parameters()]
    for _ in range(2):                                              # (the first call may set a library up)
        out = BlockFn.apply(plan, x, low, None, *plan.norm_params, *plan.weight_params)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        grads = torch.autograd.grad(out, leaves, dout)
        torch.cuda.synchronize()
        peak = torch.cuda.max_memory_allocated() - base - sum(g.numel() * g.element_size() for g in grads[2:])
        del out, grads
    assert peak <= 23 * x.numel() * x.element_size(), peak / (x.numel() * x.element_size())


def test_backward_under_autocast(dev):
    """loss.backward() inside a region of autocast, the forward outside: the row kernels read their operands' own type.  The blocks' gradients see autocast
    only through the head's products (bf16: 2^-8 an operand)."""
    import matmulfreellm_amd as mm
    torch.manual_seed(37)
    model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=200, hidden_size=256, num_hidden_layers=2)).to(dev).train()
    ids = torch.randint(0, 200, (2, 65), device=dev)
    grads = []
    for enabled in (False, True):
        model.zero_grad(set_to_none=True)
        loss = model(input_ids=ids, labels=ids).loss
        with torch.autocast("cuda", torch.bfloat16, enabled=enabled):
            loss.backward()
        grads.append({n: p.grad.double() for n, p in model.named_parameters()})
    for name, want in grads[0].items():
        assert ((grads[1][name] - want).norm() / want.norm()).item() < 1e-2, name
