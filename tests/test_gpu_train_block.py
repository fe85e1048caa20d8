"""A training step with whole blocks as autograd ops against the op-by-op composition (which a hook anywhere in the model
brings back): same loss bit for bit, gradients within rounding.  Widths on both sides of the row kernels' passes, row
counts below and above their grid, masks, frozen weights, no lower bounds."""
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
