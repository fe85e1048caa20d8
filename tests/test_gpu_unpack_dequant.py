"""The ternary weights as a dense matrix, at the edges of the vectors, the row groups, the packed blocks and the segments."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dequantised(pw, dtype):
    """[N, K], stored [K, N]."""
    from matmulfreellm_amd import _lib as L
    w = torch.empty(pw.k, pw.n, dtype=dtype, device=pw.packed.device)
    L.check(L.load().mmf_unpack_dequant_t(pw.packed.data_ptr(), pw.wdeq.data_ptr(), pw.seg_rows, pw.n, pw.k, w.data_ptr(), L.dtype_id(dtype),
                                          L.stream()), "mmf_unpack_dequant_t")
    return w.t()


@pytest.mark.parametrize("n,k,seg", [(1, 4, 1), (7, 100, 7), (33, 131, 33), (96, 1024, 32), (40, 2056, 20), (64, 4100, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_dense_weights_equal_unpacked_codes_times_scale(dev, n, k, seg, dtype):
    import matmulfreellm_amd.functional as F
    torch.manual_seed(n + k)
    pw = F.ternarize_pack(torch.randn(n, k, device=dev))
    codes = F.unpack_ternary(pw).float()
    pw.wdeq, pw.seg_rows = torch.rand(-(-n // seg), device=dev) + 0.5, seg
    scale = pw.wdeq.repeat_interleave(seg)[:n].view(n, 1)
    assert torch.equal(_dequantised(pw, dtype), (codes * scale).to(dtype))


@pytest.mark.parametrize("rows,k,norms", [(3, 1024, 1), (5, 1028, 3), (2, 2048, 3), (1100, 260, 1), (3, 4096, 3), (3, 4100, 1), (2, 6148, 1), (2, 8192, 1)])
def test_chained_norm_backward_equals_autograd(dev, rows, k, norms):
    """norm behind norm against torch autograd of the same ops in fp64 (straight through the quantiser), for each split of a row."""
    from matmulfreellm_amd.autograd import CHAIN_NORM, _chain_bwd
    torch.manual_seed(k)
    x, dres = torch.randn(rows, k, device=dev), torch.randn(rows, k, device=dev)
    w1, w2 = torch.rand(k, device=dev) + 0.5, [torch.rand(k, device=dev) + 0.5 for _ in range(norms)]
    dy = [torch.randn(rows, k, device=dev) for _ in range(norms)]
    dx, _, _, dw = _chain_bwd(CHAIN_NORM, x, None, w1, 1e-6, w2, 1e-6, dy, dres=dres)
    leaf = [t.double().requires_grad_() for t in (x, w1, *w2)]
    norm = lambda v, w: v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-6) * w
    s = norm(leaf[0], leaf[1])
    ref = torch.autograd.grad([norm(s, w) for w in leaf[2:]], leaf, [d.double() for d in dy])
    for got, want in zip((dx - dres, *dw), ref):
        assert (got.double() - want).norm() <= 2e-6 * want.norm()


@pytest.mark.parametrize("n,k,seg", [(1, 1, 1), (9, 17, 4), (31, 129, 31), (256 * 8 + 8, 144, 1024), (72, 260, 24)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_both_layouts_of_the_dense_weights_hold_the_same_values(dev, n, k, seg, dtype):
    """[N, K] and [K, N], at the edges of the row vectors, the workgroups' columns, the 16-input pieces and the segments."""
    import matmulfreellm_amd._lib as L
    import matmulfreellm_amd.functional as F
    torch.manual_seed(n * k)
    pw = F.ternarize_pack(torch.randn(n, k, device=dev))
    pw.wdeq, pw.seg_rows = torch.rand(-(-n // seg), device=dev) + 0.5, seg
    rows = torch.full((n, k), float("nan"), dtype=dtype, device=dev)
    with L.on(dev):
        L.check(L.load().mmf_unpack_dequant(pw.packed.data_ptr(), pw.wdeq.data_ptr(), seg, n, k, rows.data_ptr(), L.dtype_id(dtype),
                                            L.stream()), "mmf_unpack_dequant")
        columns = _dequantised(pw, dtype)
    assert columns.t().is_contiguous() and torch.equal(rows, columns)


@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 65), (64, 64), (72, 8), (130, 264), (1031, 33), (1024, 2048)])
def test_transpose_of_16_bit_elements(dev, rows, cols):
    """Whole and partial tiles, both widths of access, and a matrix that begins off a 16-byte boundary; nothing written past the end."""
    import matmulfreellm_amd._lib as L
    for off in (0, 1):
        x = torch.randint(-32768, 32767, (rows * cols + off,), dtype=torch.int16, device=dev)[off:].view(rows, cols)
        out = torch.full((rows * cols + 8,), 77, dtype=torch.int16, device=dev)
        L.check(L.load().mmf_transpose16(x.data_ptr(), rows, cols, out.data_ptr(), L.stream()), "mmf_transpose16")
        assert torch.equal(out[:rows * cols].view(cols, rows), x.t()) and bool((out[rows * cols:] == 77).all())


@pytest.mark.parametrize("m,n,k", [(1023, 16384, 64), (1024, 16384, 64), (1025, 16390, 70), (1088, 16390, 70), (3000, 16384, 64), (3004, 16384, 64)])
def test_weight_gradient_of_a_vocabulary_is_the_product(dev, m, n, k):
    """Both sides of the lines where the inputs are transposed first; bf16 products summed in fp32: half an ulp of the result and m roundings of the sum."""
    from matmulfreellm_amd.autograd import _weight_grad
    torch.manual_seed(m)
    d, y = torch.randn(m, n, device=dev).bfloat16(), torch.randn(m, k, device=dev).bfloat16()
    want = d.t().double() @ y.double()
    bound = want.abs() * 2 ** -8 + (d.t().double().abs() @ y.double().abs()) * m * 2 ** -24
    assert bool(((_weight_grad(d, y).double() - want).abs() <= bound).all())


@pytest.mark.parametrize("n,k,seg", [(1, 4, 1), (33, 132, 33), (96, 1024, 32)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_dense_weights_are_stored_as_their_product_takes_least_time(dev, n, k, seg, dtype):
    """The training products' weights: contraction (N) contiguous in 16 bits, rows as the packed ones in single precision; same values."""
    import matmulfreellm_amd.functional as F
    from matmulfreellm_amd.autograd import _dense_weight
    torch.manual_seed(n + k)
    pw = F.ternarize_pack(torch.randn(n, k, device=dev))
    codes = F.unpack_ternary(pw).float()
    pw.wdeq, pw.seg_rows = torch.rand(-(-n // seg), device=dev) + 0.5, seg
    w = _dense_weight(pw, dtype)
    assert (w if dtype == torch.float32 else w.t()).is_contiguous()
    assert torch.equal(w, (codes * pw.wdeq.repeat_interleave(seg)[:n].view(n, 1)).to(dtype))
