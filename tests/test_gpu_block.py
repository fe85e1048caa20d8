"""The native block call against the module path it stands for, bit for bit: row counts on both sides of every switch (one
launch per BitLinear, quantiser + contraction, swiglu epilogue), one token on a kept state, masks, inner norms that agree
or differ, stacked segments that no tile width divides.  A hook anywhere in a block makes the model take the module path."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def build(dev, dtype, hidden, trained, layers=3):
    import matmulfreellm_amd as mm
    torch.manual_seed(3)
    model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=500, hidden_size=hidden, num_hidden_layers=layers, bos_token_id=None,
                                                   eos_token_id=None))
    with torch.no_grad():
        for name, p in model.named_parameters():
            if trained and "norm" in name:
                p.copy_(0.5 + torch.rand(p.shape))
            if name.endswith("lower_bounds"):
                p.copy_(torch.randn(p.shape))
    return model.to(dev, dtype).eval()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hidden,trained", [(160, True), (512, True), (160, False)])
def test_native_block_equals_the_module_path(dev, dtype, hidden, trained):
    model = build(dev, dtype, hidden, trained)
    with torch.no_grad():
        for b, t, masked in [(1, 1, False), (1, 5, False), (2, 4, True), (3, 3, False), (1, 77, False), (3, 100, True), (2, 257, False)]:
            ids = torch.randint(0, 500, (b, t), device=dev)
            mask = (torch.arange(t, device=dev) >= torch.arange(b, device=dev).view(-1, 1) % t).long() if masked else None
            step = torch.randint(0, 500, (b, 1), device=dev)
            got = {}
            for path in ("native", "modules"):
                hooks = [layer.attn.g_norm.register_forward_hook(lambda *a: None) for layer in model.model.layers] \
                    if path == "modules" else []
                out = model(input_ids=ids, attention_mask=mask, use_cache=True, output_hidden_states=masked)
                first = [s[-1].clone() for s in out.past_key_values]
                nxt = model(input_ids=step, past_key_values=out.past_key_values, use_cache=True)
                keep = torch.ones_like(step)
                keep[0] = 0
                last = model(input_ids=step, attention_mask=keep, past_key_values=nxt.past_key_values, use_cache=True)
                got[path] = [out.logits, *first, nxt.logits, last.logits, *(s[-1] for s in last.past_key_values),
                             *(out.hidden_states or ())]
                for h in hooks:
                    h.remove()
            for i, (a, r) in enumerate(zip(got["native"], got["modules"])):
                assert torch.equal(a, r), (b, t, masked, i)


@pytest.mark.parametrize("hooked", [(0,), (1,), (2,), (3,), (4,), (1, 2), (1, 3)])
def test_what_a_hook_has_kept_is_not_written(dev, hooked):
    """Forward hooks on some layers keep their inputs and outputs (activation capture): the blocks behind them, native calls that
    reuse each other's buffers, leave those tensors as the hooks saw them."""
    model = build(dev, torch.bfloat16, 160, True, layers=6)
    ids = torch.randint(0, 500, (2, 20), device=dev)
    with torch.no_grad():
        want = model(input_ids=ids, output_hidden_states=True).hidden_states
        kept = []
        for i in hooked:
            model.model.layers[i].register_forward_hook(lambda m, args, out, i=i: kept.append((i, args[0], out[0])))
        logits = model(input_ids=ids).logits
        again = model(input_ids=ids, output_hidden_states=True)
    assert [i for i, _, _ in kept] == list(hooked) * 2
    for i, x, y in kept[:len(hooked)]:
        assert torch.equal(x, want[i]) and torch.equal(y, want[i + 1]), i
    assert torch.equal(logits, again.logits)


def test_changed_modules_are_seen(dev, monkeypatch):
    """What the module path would refuse or run differently, changed after a first forward: the mode, a module's class, a class's
    forward."""
    import matmulfreellm_amd as mm
    model = build(dev, torch.bfloat16, 160, True)
    ids = torch.randint(0, 500, (1, 20), device=dev)
    run = lambda: model(input_ids=ids).logits
    with torch.no_grad():
        want = run()
        attn, mlp = model.model.layers[1].attn, model.model.layers[1].mlp
        attn.mode = "chunk"
        with pytest.raises(NotImplementedError):
            run()
        attn.mode = "fused_recurrent"
        assert torch.equal(run(), want)

        class Double(mm.HGRNBitMLP):
            def forward(self, *args, **kwargs):
                return super().forward(*args, **kwargs) * 2

        mlp.__class__ = Double
        assert not torch.equal(run(), want)
        mlp.__class__ = mm.HGRNBitMLP
        assert torch.equal(run(), want)
        with monkeypatch.context() as patch:
            patch.setattr(mm.HGRNBitMLP, "forward", lambda self, x, residual=None, pre_norm=None: x)
            assert not torch.equal(run(), want)
        assert torch.equal(run(), want)


def test_a_parametrised_weight_is_packed_anew(dev):
    """A weight behind a parametrisation is another tensor on each access, often at the same address; its own tensor changes here."""
    model = build(dev, torch.bfloat16, 160, True)
    ids = torch.randint(0, 500, (1, 20), device=dev)
    run = lambda: model(input_ids=ids).logits
    with torch.no_grad():
        want, mlp = run(), model.model.layers[1].mlp

        class Scale(torch.nn.Module):
            def __init__(self):
                super().__init__()
                self.s = torch.nn.Parameter(torch.ones((), device=dev, dtype=torch.bfloat16))

            def forward(self, w):
                return w * self.s

        scale = Scale()
        torch.nn.utils.parametrize.register_parametrization(mlp.down_proj, "weight", scale)
        assert torch.equal(run(), want)
        scale.s.fill_(-1.0)
        assert not torch.equal(run(), want)
        mlp.down_proj.parametrizations.weight.original.neg_()
        assert torch.equal(run(), want)


def test_a_written_or_replaced_parameter_is_seen(dev):
    model = build(dev, torch.bfloat16, 160, True)
    ids = torch.randint(0, 500, (1, 20), device=dev)
    attn = model.model.layers[1].attn
    with torch.no_grad():
        logits = [model(input_ids=ids).logits]
        attn.f_proj.norm.weight.mul_(1.5)
        logits.append(model(input_ids=ids).logits)
        attn.o_proj.weight = torch.nn.Parameter(torch.randn_like(attn.o_proj.weight))
        logits.append(model(input_ids=ids).logits)
        attn.g_norm.eps = 0.5
        logits.append(model(input_ids=ids).logits)
        hook = attn.g_norm.register_forward_hook(lambda *a: None)
        assert torch.equal(logits[-1], model(input_ids=ids).logits)
        hook.remove()
    assert not any(torch.equal(a, b) for a, b in zip(logits, logits[1:]))


@pytest.mark.parametrize("after", ["prompt", "training step", "generate"])
def test_a_model_that_has_run_can_be_copied_and_saved_whole(dev, after):
    import copy
    import io
    model = build(dev, torch.bfloat16, 160, True)
    ids = torch.randint(0, 500, (2, 20), device=dev)
    if after == "training step":
        model.train()(input_ids=ids, labels=ids).loss.backward()
        model.eval()
    with torch.no_grad():
        if after == "generate":
            model.generate(ids, max_new_tokens=4)
        want, tokens = model(input_ids=ids).logits, model.generate(ids, max_new_tokens=4) if after == "generate" else None
        buf = io.BytesIO()
        torch.save(model, buf)
        buf.seek(0)
        for other in (copy.deepcopy(model), torch.load(buf, weights_only=False)):
            assert torch.equal(other(input_ids=ids).logits, want)
            if tokens is not None:
                assert torch.equal(other.generate(ids, max_new_tokens=4), tokens)
            other.model.layers[1].attn.g_norm.eps = 0.5
            other.model.layers[1].mlp.down_proj.weight.neg_()
            changed = other(input_ids=ids).logits
            other.model.layers[0].attn.g_norm.register_forward_hook(lambda *a: None)
            assert torch.equal(other(input_ids=ids).logits, changed) and not torch.equal(changed, want)
        assert torch.equal(model(input_ids=ids).logits, want)


def test_a_dropped_model_gives_its_memory_back(dev):
    """After prompts, a training step and generation through the captured graphs and the resident launch, with the cycle collector off."""
    import gc
    held = []
    gc.collect()
    gc.disable()
    try:
        for use in (lambda m, ids: m(input_ids=ids), lambda m, ids: m(input_ids=ids, labels=ids).loss.backward(),
                    lambda m, ids: m.generate(ids, max_new_tokens=3), lambda m, ids: m.generate(ids[:1], max_new_tokens=3)):
            before = torch.cuda.memory_allocated(dev)
            model, ids = build(dev, torch.bfloat16, 512, True), torch.randint(0, 500, (2, 20), device=dev)
            weights = sum(p.numel() * p.element_size() for p in model.parameters())
            with torch.set_grad_enabled("backward" in use.__code__.co_names):
                use(model, ids)
            torch.cuda.synchronize(dev)
            del model, ids
            held.append((torch.cuda.memory_allocated(dev) - before) / weights)
    finally:
        gc.enable()
    assert max(held) < 0.2, held
