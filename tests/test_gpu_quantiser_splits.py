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


@pytest.mark.parametrize("m,k", [(193, 4), (193, 2048), (391, 8192), (513, 132), (515, 2048), (700, 5632), (1281, 1024), (2100, 516), (2100, 260)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_codes_stored_through_lds_lie_where_row_major_codes_say(dev, m, k, dtype):
    """Two, four and eight rows a workgroup, a last workgroup with rows past the end, a grid past, at and short of whole groups of 64 workgroups,
    inputs past k: tiled codes against the row kernel's row-major ones, and nothing written behind the last block of rows."""
    import matmulfreellm_amd.functional as F
    torch.manual_seed(m + k)
    L, lib = F.L, F.L.load()
    x = torch.randn(m, k, device=dev).to(dtype)
    w1, *nw = [(torch.rand(k, device=dev) + 0.5).to(dtype) for _ in range(4)]
    size, dt = lib.mmf_codes_bytes(m, k, 1), L.dtype_id(dtype)
    q = torch.full((3 * size + 64,), 77, dtype=torch.int8, device=dev)
    deq, qsum = torch.empty(3, m, device=dev), torch.empty(3, m, dtype=torch.int32, device=dev)
    normed = F.rmsnorm(x, w1, eps=1e-6)

    def same(j, v):
        codes, d, s = F.rmsnorm_quant(v, nw[j], eps=1e-8, tiled=False)
        assert torch.equal(F.codes_tiled_to_rowmajor(q[j * size:(j + 1) * size], m, k), codes.view(m, -1)[:, :k])
        assert torch.equal(deq[j], d) and torch.equal(qsum[j], s)

    L.check(lib.mmf_rmsnorm_quant_multi(x.data_ptr(), k, w1.data_ptr(), 1e-6, *(w.data_ptr() for w in nw), 1e-8, q.data_ptr(), deq.data_ptr(),
                                        qsum.data_ptr(), m, k, dt, dt, L.stream()), "multi")
    for j in range(3):
        same(j, normed)
    assert bool((q[3 * size:] == 77).all())
    q.fill_(77)
    L.check(lib.mmf_rmsnorm_quant_fused(0, x.data_ptr(), k, None, 0, None, 0, None, None, 0.0, nw[0].data_ptr(), 1e-8, None, None, q.data_ptr(),
                                        deq.data_ptr(), qsum.data_ptr(), m, k, dt, dt, L.stream()), "plain")
    same(0, x)
    rows = q[:size].view(-1, (k + 127) // 128 * 8, 32, 16)
    assert bool((rows[m // 32, :, m % 32:] == 77).all()) and bool((q[size:] == 77).all())
