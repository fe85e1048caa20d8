"""Which kernels a contraction's rows take, and where they are cut: the tests of cut rows and of narrow tiles rely on it, and segments with codes of their
own whose columns do not suit the tiles are never cut (each launch of theirs is one a segment already)."""
import ctypes

import pytest

TILE_COLUMNS = {5: 32, 16: 256, 17: 512, 18: 256, 19: 128}


def plan(m, k, n, seg=0, swiglu=0):
    """(rows of the first launch, its kernel, the second one's or -1)"""
    from matmulfreellm_amd import _lib as L
    first, configs = ctypes.c_int64(), (ctypes.c_int * 2)()
    assert L.load().mmf_bitlinear_mfma_plan(m, k, n, seg, swiglu, ctypes.byref(first), configs) == 0
    return first.value, configs[0], configs[1]


def test_plans_of_known_shapes():
    assert plan(1, 2048, 2048) == (1, 5, -1)
    assert plan(16384, 2048, 2048)[1:] == (17, -1)
    assert plan(1377, 2048, 6144) == (1344, 17, 5)
    assert plan(1001, 5632, 2048) == (1001, 19, -1)


@pytest.mark.parametrize("d", [512, 640, 768, 1024, 1152, 1312, 1536, 2048, 2304, 2560])
def test_segments_are_cut_only_where_every_launch_suits_them(d):
    cut = 0
    for m in range(65, 6000, 7):
        first, *configs = plan(m, d, 3 * d, d)
        if first < m:
            cut += 1
            assert first % 64 == 0 and m - first <= 320
            assert all(d % TILE_COLUMNS[c] == 0 for c in configs), (m, first, configs)
    assert cut or d not in (1024, 1536, 2048, 2560)
    assert not cut or d % 128 == 0
    assert any(plan(m, d, 3 * d)[0] < m for m in range(65, 6000, 7)) or d == 768       # with one set of codes nearly all are cut somewhere


def test_shapes_that_are_none_are_refused():
    from matmulfreellm_amd import _lib as L
    first, configs = ctypes.c_int64(), (ctypes.c_int * 2)()
    for m, k, n, seg in ((0, 1, 1, 0), (1, 0, 1, 0), (1, 1, 0, 0), (1, 1, 1, -1), (1, 1, 1 << 31, 0)):
        assert L.load().mmf_bitlinear_mfma_plan(m, k, n, seg, 0, ctypes.byref(first), configs) < 0
