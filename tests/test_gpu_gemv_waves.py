"""The fused GEMV at the edges of its wave counts: rows that just fill or just overflow 4 and 8 waves, and one more workgroup than CUs,
against the quantiser + matrix-core pair of launches (bit for bit), with and without prologue, addend and epilogue."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [96, 1020, 1024, 1028, 2048, 2052])
@pytest.mark.parametrize("m,n", [(1, 64), (4, 2048), (5, 2048), (8, 1056)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gemv_equals_quantiser_and_contraction(dev, m, n, k, dtype):
    import matmulfreellm_amd.functional as F
    torch.manual_seed(k + n)
    pw = F.ternarize_pack(torch.randn(n, k, device=dev).to(dtype))
    x, add = torch.randn(m, k, device=dev).to(dtype), torch.randn(m, n, device=dev).to(dtype)
    w = (torch.rand(k, device=dev) + 0.5).to(dtype)
    assert torch.equal(F.bitlinear(x, w, pw, path="gemv"), F.bitlinear(x, w, pw, path="mfma"))
    assert torch.equal(F.bitlinear(x, w, pw, path="gemv", addend=add), F.bitlinear(x, w, pw, path="mfma", addend=add))


@pytest.mark.parametrize("hidden", [1024, 1152, 2048])
@pytest.mark.parametrize("batch", [2, 5, 8])
@pytest.mark.parametrize("trained", [False, True])
def test_decode_chain_equals_the_batch_1_rows(dev, hidden, batch, trained):
    import matmulfreellm_amd as mm
    torch.manual_seed(hidden)
    model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=512, hidden_size=hidden, num_hidden_layers=2)).to(dev, torch.bfloat16).eval()
    if trained:
        for p in model.parameters():
            if p.dim() == 1:
                p.data.uniform_(0.5, 1.5)
    ids = torch.randint(0, 512, (batch, 7), device=dev)
    got = model.generate(ids, max_new_tokens=6)
    for r in range(batch):
        assert torch.equal(got[r:r + 1], model.generate(ids[r:r + 1], max_new_tokens=6)), r
