"""The largest logit's lowest index: one and several passes over a row, ragged and strided rows, ties across threads and passes, NaN, infinities."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v,ld", [(1, 1), (7, 9), (500, 500), (32000, 32000), (32767, 32769), (32768, 32768), (32776, 32776), (100003, 100003)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_argmax(dev, v, ld, dtype):
    from matmulfreellm_amd import _lib as L
    torch.manual_seed(v)
    wide = (torch.randn(9, ld, device=dev) * 3).to(dtype)
    x = wide[:, :v]
    x[1] = 2.0                                                    # every element ties
    x[2, v // 2:] = 30.0
    x[3, 0] = float("nan")
    x[4] = float("nan")
    x[5] = float("-inf")
    x[6, : v // 2] = float("nan")
    x[6, v // 2:] = float("-inf")
    x[7, -1] = float("inf")
    x[8] = -0.0
    x[8, v // 3:] = 0.0
    out = torch.full((9,), -1, dtype=torch.int64, device=dev)
    L.check(L.load().mmf_argmax(x.data_ptr(), ld, 9, v, out.data_ptr(), L.dtype_id(dtype), L.stream()), "mmf_argmax")
    want = []
    for row in x.float().cpu():
        top = row[~row.isnan()]
        want.append(int((row == top.max()).nonzero()[0, 0]) if len(top) else 0)
    assert out.tolist() == want
