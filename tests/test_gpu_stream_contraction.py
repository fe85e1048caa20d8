"""The weight-stream contraction at the edges of its variants: one to four k-blocks per wave of 16 and of 8, the last one missing
in some waves, ragged rows and columns, segments with codes of their own, and its swiglu form -- against the exact integer
contraction of the oracle's packing and the tiled kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(dev, m, k, n, sets=1, seed=1):
    import matmulfreellm_amd.functional as F
    torch.manual_seed(seed)
    pw = F.ternarize_pack(torch.randn(n, k, device=dev).bfloat16())
    lib = F.L.load()
    q = torch.zeros(sets, lib.mmf_codes_bytes(m, k, 1), dtype=torch.int8, device=dev)
    codes, deq, qsum = [], [], []
    for s in range(sets):
        x = torch.randn(m, k, device=dev).bfloat16()
        qs = F.rmsnorm_quant(x, torch.ones(k, device=dev).bfloat16(), tiled=True)
        q[s].copy_(qs[0])
        codes.append(F.codes_tiled_to_rowmajor(qs[0], m, k).cpu().long())
        deq.append(qs[1])
        qsum.append(qs[2])
    return F, lib, pw, q, codes, torch.stack(deq), torch.stack(qsum)


def exact(F, pw, codes, deq, dtype):
    acc = codes @ F.unpack_ternary(pw).cpu().long().t()
    return (acc.float() * deq.cpu().view(-1, 1) * pw.wdeq.cpu()[0]).to(dtype)


@pytest.mark.parametrize("m,k,n", [(1, 128, 32), (33, 1920, 40), (64, 2048, 2048), (64, 2176, 2048), (64, 5632, 2048), (70, 8192, 1056),
                                   (64, 1024, 5600), (64, 2048, 6144), (40, 3968, 4128), (33, 8192, 4160)])
def test_stream_contraction_is_exact(dev, m, k, n):
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, n)
    out = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, torch.bfloat16, config=5)
    assert torch.equal(out.cpu(), exact(F, pw, codes[0], deq[0], torch.bfloat16))


@pytest.mark.parametrize("m,k,inter", [(9, 160, 512), (64, 2048, 5632), (77, 1024, 2816), (33, 8192, 96)])
def test_stream_swiglu_equals_contraction_then_swiglu(dev, m, k, inter):
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, 2 * inter, seed=2)
    y = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, torch.bfloat16)
    assert torch.equal(F.bitlinear_mfma_swiglu(q[0], deq[0], qsum[0], pw, m, torch.bfloat16), F.swiglu(y[:, :inter], y[:, inter:]))


@pytest.mark.parametrize("m,k,seg,config", [(40, 512, 96, -1), (64, 2048, 2048, -1), (300, 512, 96, -1), (600, 512, 512, 17), (600, 512, 160, 17)])
def test_segments_contract_their_own_codes(dev, m, k, seg, config):
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, 3 * seg, sets=3, seed=3)
    pw.wdeq, pw.seg_rows = pw.wdeq.repeat(3) * torch.tensor([1.0, 2.0, 0.5], device=dev), seg
    out = torch.empty(m, 3 * seg, dtype=torch.bfloat16, device=dev)
    F.L.check(lib.mmf_bitlinear_mfma_multi(q.data_ptr(), q.stride(0), deq.data_ptr(), qsum.data_ptr(), pw.packed.data_ptr(),
                                           pw.wdeq.data_ptr(), seg, out.data_ptr(), 3 * seg, m, k, 3 * seg, 1, config, F.L.stream()), "multi")
    for s in range(3):
        alone = F.bitlinear_mfma(q[s], deq[s], qsum[s], pw, m, torch.bfloat16)
        assert torch.equal(out[:, s * seg:(s + 1) * seg], alone[:, s * seg:(s + 1) * seg]), s
