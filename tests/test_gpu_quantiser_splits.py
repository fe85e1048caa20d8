"""The fused quantisers where their split changes: rows per workgroup (192, 512, 1280 rows) and passes per row, full and ragged last
passes, against the unfused norm -> quantise launches (bit for bit)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 1024, 1028, 2048, 2820, 3076, 4096, 5632])
@pytest.mark.parametrize("m", [192, 193, 513, 1281])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_fused_quantisers_equal_norm_then_quantise(dev, m, k, dtype):
    import matmulfreellm_amd.functional as F
    torch.manual_seed(k)
    n = 32
    pw = F.ternarize_pack(torch.randn(n, k, device=dev).to(dtype))
    x, a = torch.randn(m, k, device=dev).to(dtype), torch.randn(m, k, device=dev).to(dtype)
    x[3] = 0
    w1, w2 = (torch.rand(k, device=dev) + 0.5).to(dtype), (torch.rand(k, device=dev) + 0.5).to(dtype)
    plain = lambda v: F.bitlinear(v, w2, pw, path="mfma")
    from matmulfreellm_amd.layernorm import rms_norm_fn
    from matmulfreellm_amd.fused_norm_gate import rms_norm_swish_gate_fn
    normed = rms_norm_fn(x, w1, None, eps=1e-6)
    assert torch.equal(F.bitlinear(x, w2, pw, prologue=("norm", w1, 1e-6)), plain(normed))
    normed, res = rms_norm_fn(x, w1, None, residual=a, eps=1e-6, prenorm=True)
    out, res2 = F.bitlinear(x, w2, pw, prologue=("resnorm", a, w1, 1e-6))
    assert torch.equal(out, plain(normed)) and torch.equal(res, res2)
    assert torch.equal(F.bitlinear(x, w2, pw, prologue=("swiglu", a)), plain(F.swiglu(x, a)))
