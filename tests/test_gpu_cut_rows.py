"""Contractions whose last rows take a launch of their own: the bits of one launch (a fixed tile shape, itself held to the oracle in
test_gpu_ops.py), with one row and with many behind the last whole round, a residual, a bias, a wider output and codes of its own per segment."""
import pytest
import torch

from test_contraction_plan import plan

pytestmark = pytest.mark.gpu


def _operands(dev, m, k, n, dtype, segments=1):
    import matmulfreellm_amd.functional as F_
    from matmulfreellm_amd import _lib as L
    torch.manual_seed(m + n)
    w = F_.ternarize_pack((torch.randn(n, k, device=dev) * 0.02).to(torch.bfloat16))
    stride = L.load().mmf_codes_bytes(m, k, 1)
    q = torch.randint(-127, 128, (segments * stride,), dtype=torch.int8, device=dev)
    deq = torch.rand(segments, m, device=dev) + 0.01
    qsum = torch.randint(-5000, 5000, (segments, m), dtype=torch.int32, device=dev)
    wdeq = torch.rand(segments, device=dev) + 0.01
    return L, L.load(), w, stride, q, deq, qsum, wdeq


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("m,k,n,pad,extra", [(1345, 2048, 6144, 0, None), (1377, 2048, 6112, 64, None), (1449, 2048, 6144, 0, "bias"),
                                             (2096, 5632, 2048, 0, "addend"), (2096, 5632, 2048, 16, "addend"), (2743, 1024, 3072, 0, None)])
def test_rows_in_two_launches(dev, dtype, m, k, n, pad, extra):
    assert plan(m, k, n)[0] < m
    L, lib, w, _, q, deq, qsum, wdeq = _operands(dev, m, k, n, dtype)
    other = torch.randn(m, n + pad, device=dev).to(dtype)
    bias = torch.randn(n, device=dev).to(dtype)

    def run(config):
        out = torch.zeros(m, n + pad, dtype=dtype, device=dev)
        rc = lib.mmf_bitlinear_mfma(q.data_ptr(), deq.data_ptr(), qsum.data_ptr(), w.packed.data_ptr(), wdeq.data_ptr(), w.seg_rows,
                                    bias.data_ptr() if extra == "bias" else None, other.data_ptr() if extra == "addend" else None,
                                    out.data_ptr(), n + pad, m, k, n, L.dtype_id(dtype), config, L.stream())
        assert rc == 0
        return out

    got = run(-1)
    assert torch.equal(got, run(17)) and torch.equal(got, run(18))
    assert not pad or not got[:, n:].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,k,n,seg", [(1377, 2048, 6144, 2048), (1345, 2048, 6144, 2048), (1093, 2560, 7680, 2560), (2743, 1024, 3072, 1024)])
def test_segments_with_codes_of_their_own(dev, dtype, m, k, n, seg):
    assert plan(m, k, n, seg)[0] < m
    L, lib, w, stride, q, deq, qsum, wdeq = _operands(dev, m, k, n, dtype, n // seg)

    def run(config):
        out = torch.zeros(m, n, dtype=dtype, device=dev)
        rc = lib.mmf_bitlinear_mfma_multi(q.data_ptr(), stride, deq.data_ptr(), qsum.data_ptr(), w.packed.data_ptr(), wdeq.data_ptr(), seg,
                                          out.data_ptr(), n, m, k, n, L.dtype_id(dtype), config, L.stream())
        assert rc == 0
        return out

    assert torch.equal(run(-1), run(18))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("m,k,n", [(715, 2048, 11264), (705, 2048, 11264), (3066, 2048, 11264), (1848, 2560, 13824)])
def test_swiglu_rows_in_two_launches(dev, dtype, m, k, n):
    """Against launches of 128 rows each, which are not cut."""
    assert plan(m, k, n, 0, 1)[0] < m and plan(128, k, n, 0, 1)[0] == 128
    L, lib, w, _, q, deq, qsum, wdeq = _operands(dev, m, k, n, dtype)
    deq *= 1e-3                                                     # gates in the sigmoid's range

    def run(out, r, rows):
        rc = lib.mmf_bitlinear_mfma_swiglu(q.data_ptr() + r * k, deq.data_ptr() + 4 * r, qsum.data_ptr() + 4 * r, w.packed.data_ptr(), wdeq.data_ptr(),
                                           w.seg_rows, out[r:].data_ptr(), n // 2, rows, k, n, L.dtype_id(dtype), L.stream())
        assert rc == 0

    got, want = (torch.zeros(m, n // 2, dtype=dtype, device=dev) for _ in range(2))
    run(got, 0, m)
    for r in range(0, m, 128):
        run(want, r, min(128, m - r))
    assert torch.equal(got, want)
