"""Gate math and recurrence in one launch against the two launches it stands for (bit for bit): around the lengths of its tiles for each
width of a workgroup's columns, ragged columns, masks, lower bounds, states, strided operands."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,d", [(1, 16), (2, 40), (3, 1024), (3, 4096), (5, 2080), (9, 4096)])
@pytest.mark.parametrize("t", [1, 9, 10, 29, 30, 31, 60, 61, 119, 120, 121, 240, 367, 512, 513])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_gate_scan_equals_gate_then_scan(dev, b, d, t, dtype):
    import matmulfreellm_amd.functional as F
    torch.manual_seed(t)
    ifg = torch.randn(b * t, 3 * d, device=dev).to(dtype)
    i, f = ifg[:, :d], ifg[:, d:2 * d]
    lb, h0 = torch.rand(d, device=dev) * 0.5, torch.randn(b, 1, d, device=dev)
    mask = (torch.rand(b * t, device=dev) > 0.2).to(torch.uint8)
    for use_lb, use_mask, use_h0 in itertools.product((True, False), repeat=3):
        x, g = F.hgrn_gate(i, f, lb if use_lb else None, mask if use_mask else None)
        want, last = F.hgrn_recurrent(x.view(b, 1, t, d), g.view(b, 1, t, d), h0 if use_h0 else None, True)
        o, ht = torch.empty(b * t, d, dtype=dtype, device=dev), torch.empty(b, d, device=dev)
        F.L.check(F.L.load().mmf_hgrn_gate_scan(i.data_ptr(), 3 * d, f.data_ptr(), 3 * d, F.L.ptr(lb) if use_lb else None,
                                                F.L.ptr(mask) if use_mask else None, F.L.ptr(h0) if use_h0 else None, o.data_ptr(),
                                                ht.data_ptr(), b, t, d, F.L.dtype_id(dtype), F.L.stream()), "gate_scan")
        assert torch.equal(o.view(b, t, d), want.view(b, t, d)) and torch.equal(ht, last.view(b, d))


# single channels (odd widths and strides) and pairs; rows of 256 KiB, whose bases move every 16 tiles (of 120 steps), and more
@pytest.mark.parametrize("b,t,d,ld", [(2, 130, 41, 123), (1, 65, 40, 121), (3, 700, 34, 102), (1, 4100, 16, 131072), (2, 2161, 18, 131072), (1, 300, 32, 131072),
                                      (1, 130, 32, 140000), (9, 2100, 128, 32768)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_single_channels_and_pairs(dev, b, t, d, ld, dtype):
    import matmulfreellm_amd.functional as F
    torch.manual_seed(t)
    if dtype == torch.float32 and ld > 100000:
        ld //= 2
    wide = torch.randn(b * t, ld, device=dev).to(dtype)
    i, f = wide[:, :d], wide[:, ld - d - ld % 2:ld - ld % 2]
    lb, mask = torch.rand(d, device=dev), (torch.rand(b * t, device=dev) > 0.2).to(torch.uint8)
    x, g = F.hgrn_gate(i.contiguous(), f.contiguous(), lb, mask)
    want, last = F.hgrn_recurrent(x.view(b, 1, t, d), g.view(b, 1, t, d), None, True)
    o, ht = torch.empty(b * t, d, dtype=dtype, device=dev), torch.empty(b, d, device=dev)
    F.L.check(F.L.load().mmf_hgrn_gate_scan(i.data_ptr(), ld, f.data_ptr(), ld, F.L.ptr(lb), F.L.ptr(mask), None, o.data_ptr(), ht.data_ptr(), b, t, d,
                                            F.L.dtype_id(dtype), F.L.stream()), "gate_scan")
    assert torch.equal(o.view(b, t, d), want.view(b, t, d)) and torch.equal(ht, last.view(b, d))
