"""Quantisers where the rows a workgroup change (1024 / 1025, 1536 / 1537, 2 to 8 rows): the codes, scales and sums of launches of 96 rows, which have a
workgroup a row and are held to the oracle in test_gpu_ops.py."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,k", [(1024, 2048), (1025, 2048), (1536, 2000), (1537, 2048), (1535, 3072), (1025, 1024), (1281, 1000), (1100, 5632)])
def test_rows_a_workgroup(dev, dtype, m, k):
    from matmulfreellm_amd import _lib as L
    lib, dt = L.load(), L.dtype_id(dtype)
    torch.manual_seed(m + k)
    x, aux = (torch.randn(m, k, device=dev).to(dtype) for _ in range(2))
    w1, *nw = [(0.5 + torch.rand(k, device=dev)).to(dtype) for _ in range(4)]
    kp = -(-k // 128) * 128

    def run(pro, r, rows):
        n = 3 if pro == "multi" else 1
        q = torch.zeros(n, lib.mmf_codes_bytes(rows, k, 1), dtype=torch.int8, device=dev)
        deq, qsum, res = torch.zeros(n, rows, device=dev), torch.zeros(n, rows, dtype=torch.int32, device=dev), torch.zeros(rows, k, dtype=dtype, device=dev)
        out = (q.data_ptr(), deq.data_ptr(), qsum.data_ptr(), rows, k, dt, dt, L.stream())
        if pro == "multi":
            rc = lib.mmf_rmsnorm_quant_multi(x[r:].data_ptr(), k, w1.data_ptr(), 1e-6, *(w.data_ptr() for w in nw), 1e-6, *out)
        else:
            second = aux[r:].data_ptr() if pro in (2, 5) else None
            rc = lib.mmf_rmsnorm_quant_fused(pro, x[r:].data_ptr(), k, second, k if second else 0, None, 0, res.data_ptr() if pro == 2 else None,
                                             w1.data_ptr() if pro else None, 1e-6, nw[0].data_ptr(), 1e-6, None, None, *out)
        assert rc == 0
        return q, deq, qsum, res

    for pro in (0, 1, 2, 5, "multi"):
        q, deq, qsum, res = run(pro, 0, m)
        for r in range(0, m, 96):
            rows = min(96, m - r)
            wq, wdeq, wqsum, wres = run(pro, r, rows)
            codes = q[:, r * kp:r * kp + wq.shape[1]].view(len(q), -1, kp // 16, 32, 16)[..., :, :]
            want = wq.view(len(q), -1, kp // 16, 32, 16)
            live = (torch.arange(want.shape[1] * 32, device=dev) < rows).view(-1, 1, 32, 1)
            assert torch.equal(codes * live, want * live), (pro, r)
            assert torch.equal(deq[:, r:r + rows], wdeq) and torch.equal(qsum[:, r:r + rows], wqsum) and torch.equal(res[r:r + rows], wres), (pro, r)
