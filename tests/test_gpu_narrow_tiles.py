"""64 x 128 tiles of the tiled contraction: against the oracle at the edges of tiles, k-blocks and of one tile per CU, and where the
dispatch takes them the bits of the other tiles."""
import pytest
import torch

from test_contraction_plan import plan

pytestmark = pytest.mark.gpu


def _same(out, ref):
    return torch.equal(out.cpu(), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("m,k,n", [(65, 256, 96), (64, 256, 128), (129, 1024, 136), (300, 1000, 648), (127, 2048, 1028), (1030, 256, 2050), (1090, 512, 2050)])
def test_narrow_tiles_vs_oracle(dev, dtype, m, k, n):
    import matmulfreellm_amd.functional as F_
    from oracle import bitlinear as ob
    torch.manual_seed(m + n)
    x, w = torch.randn(m, k).to(dtype), (torch.randn(n, k) * 0.02).to(dtype)
    nw = (0.5 + torch.rand(k)).to(dtype)
    bias, addend = torch.randn(n).to(dtype), torch.randn(m, n).to(dtype)
    ref = ob.bitlinear_spec(x, w, nw, eps=1e-8)
    pw = F_.ternarize_pack(w.to(dev))
    q, deq, qsum = F_.rmsnorm_quant(x.to(dev), nw.to(dev), eps=1e-8, tiled=True)
    args = (q, deq, qsum, pw, m, dtype)
    assert _same(F_.bitlinear_mfma(*args, config=19), ref)
    for extra in ({"bias": bias.to(dev)}, {"addend": addend.to(dev)}):
        assert torch.equal(F_.bitlinear_mfma(*args, config=19, **extra), F_.bitlinear_mfma(*args, config=16, **extra))


@pytest.mark.parametrize("m,k,n", [(1001, 5632, 2048), (2002, 5632, 2048), (2400, 2048, 2048), (1600, 2816, 1024), (700, 6912, 2560), (310, 2048, 6144)])
def test_dispatch_to_narrow_tiles(dev, m, k, n):
    import matmulfreellm_amd.functional as F_
    from matmulfreellm_amd import _lib as L
    assert 19 in plan(m, k, n)[1:]
    torch.manual_seed(m)
    pw = F_.ternarize_pack((torch.randn(n, k, device=dev) * 0.02).bfloat16())
    q = torch.randint(-127, 128, (L.load().mmf_codes_bytes(m, k, 1),), dtype=torch.int8, device=dev)
    deq, qsum = torch.rand(m, device=dev), torch.randint(-5000, 5000, (m,), dtype=torch.int32, device=dev)
    got = F_.bitlinear_mfma(q, deq, qsum, pw, m, torch.bfloat16)
    assert torch.equal(got, F_.bitlinear_mfma(q, deq, qsum, pw, m, torch.bfloat16, config=17))
    assert torch.equal(got, F_.bitlinear_mfma(q, deq, qsum, pw, m, torch.bfloat16, config=19))


@pytest.mark.parametrize("seg", [640, 608])
def test_narrow_tiles_of_segments_with_codes_of_their_own(dev, seg):
    """Segments of whole tiles in one launch, others in a launch each."""
    import matmulfreellm_amd.functional as F_
    from matmulfreellm_amd import _lib as L
    m, k, n, lib = 200, 512, 3 * seg, L.load()
    torch.manual_seed(seg)
    w = F_.ternarize_pack((torch.randn(n, k, device=dev) * 0.02).bfloat16())
    stride = lib.mmf_codes_bytes(m, k, 1)
    q = torch.randint(-127, 128, (3 * stride,), dtype=torch.int8, device=dev)
    deq, wdeq = torch.rand(3, m, device=dev), torch.rand(3, device=dev)
    qsum = torch.randint(-5000, 5000, (3, m), dtype=torch.int32, device=dev)

    def run(config):
        out = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
        assert lib.mmf_bitlinear_mfma_multi(q.data_ptr(), stride, deq.data_ptr(), qsum.data_ptr(), w.packed.data_ptr(), wdeq.data_ptr(), seg,
                                            out.data_ptr(), n, m, k, n, L.dtype_id(out.dtype), config, L.stream()) == 0
        return out

    assert torch.equal(run(19), run(5))
