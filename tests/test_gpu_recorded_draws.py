"""Draws inside the decode step against the same draws made from the step's logits one by one, around the length of the recorded history;
on the launch chain, the matrix-core chain and the resident step."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 3, 12])
@pytest.mark.parametrize("steps", [1, 31, 32, 33, 64])
def test_recorded_draws_equal_single_draws(dev, batch, steps):
    import matmulfreellm_amd as mm
    import matmulfreellm_amd.functional as F
    torch.manual_seed(batch)
    model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=512, hidden_size=256, num_hidden_layers=2)).to(dev, torch.bfloat16).eval()
    eng = mm.DecodeEngine.for_model(model, batch)
    for top_p, temperature, top_k in ((0.4, 0.6, 50), (1.5, 3.0, 0)):
        u, first = torch.rand(steps, batch, device=dev), torch.randint(0, 512, (batch,), device=dev)
        eng.load_state(None)
        eng.tok.copy_(first)
        got = eng.run(steps, draw=(u, top_p, temperature, top_k))
        eng.check()
        eng.load_state(None)
        tok, want = first, [first]
        for t in range(steps):
            tok = F.sample_top_p(eng.step(tok), top_p, temperature, u[t], top_k=top_k)
            want.append(tok)
        assert torch.equal(got, torch.stack(want))
