"""Quantisers that bring the next launch's weights into the cache: the same codes, scales and sums as without, whatever the bytes (none, less than
a line, more lines than the launch has threads) and the rows a workgroup (1, 2, 4, 8); arguments that cannot be read are refused."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(9, 256), (200, 160), (300, 2048), (700, 1024), (1400, 1024), (1377, 5632), (40, 30)])
@pytest.mark.parametrize("nbytes", [0, 112, 128, 1 << 20, 3 << 24])
def test_quantisers_with_weights_ahead(dev, m, k, nbytes):
    from matmulfreellm_amd import _lib as L
    lib = L.load()
    torch.manual_seed(m + k)
    x = torch.randn(m, k, device=dev).bfloat16()
    w1, *nw = [(0.5 + torch.rand(k, device=dev)).bfloat16() for _ in range(4)]
    weights = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    ptr = weights.data_ptr() if nbytes else None

    def run(multi, *ahead):
        n = 3 if multi else 1
        out = [torch.zeros(n * lib.mmf_codes_bytes(m, k, 1), dtype=torch.int8, device=dev), torch.zeros(n, m, device=dev),
               torch.zeros(n, m, dtype=torch.int32, device=dev)]
        name = ("mmf_rmsnorm_quant_multi" if multi else "mmf_rmsnorm_quant_fused") + ("_ahead" if ahead else "")
        if multi:
            args = (x.data_ptr(), k, w1.data_ptr(), 1e-6, *(w.data_ptr() for w in nw), 1e-6)
        else:
            args = (1, x.data_ptr(), k, None, 0, None, 0, None, w1.data_ptr(), 1e-6, nw[0].data_ptr(), 1e-6, None, None)
        rc = getattr(lib, name)(*args, *(t.data_ptr() for t in out), m, k, *ahead, L.dtype_id(x.dtype), L.dtype_id(x.dtype), L.stream())
        return rc, out

    for multi in (False, True):
        rc, want = run(multi)
        assert rc == 0
        rc, got = run(multi, ptr, nbytes)
        assert rc == 0 and all(torch.equal(a, b) for a, b in zip(want, got))
        assert run(multi, ptr, -1)[0] < 0 and run(multi, x.data_ptr() + 2, 128)[0] < 0
