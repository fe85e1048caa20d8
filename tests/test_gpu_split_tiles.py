"""The tiles whose two groups of waves take alternate k-blocks, at the edges: two k-blocks (one step), a step count off the ring of
three, ragged rows and columns, the slow epilogue (bias, unaligned rows), an addend, segments, the swiglu form."""
import pytest
import torch

from test_gpu_stream_contraction import exact, operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(1, 256, 32), (65, 512, 256), (77, 768, 264), (200, 1024, 515), (1377, 2048, 2048), (2002, 5632, 1000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_split_tiles_are_exact(dev, m, k, n, dtype):
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, n)
    out = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=18)
    assert torch.equal(out.cpu(), exact(F, pw, codes[0], deq[0], dtype))
    bias, add = torch.randn(n, device=dev).to(dtype), torch.randn(m, n, device=dev).to(dtype)
    for kw in ({"bias": bias}, {"addend": add}):
        assert torch.equal(F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=18, **kw),
                           F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=16, **kw)), tuple(kw)


@pytest.mark.parametrize("blocks", range(1, 9))
def test_every_end_of_the_k_loop_is_exact(dev, blocks):
    """One to eight k-blocks, so that the loop of three ends at each of them in each of its first rounds; rows that end inside, at and behind a
    16-row fragment, columns inside one; the lean epilogue (n = 264) and the general one (n = 257)."""
    for m, n in ((15, 264), (112, 257), (145, 264)):
        F, lib, pw, q, codes, deq, qsum = operands(dev, m, 128 * blocks - 3, n, seed=blocks)
        want = exact(F, pw, codes[0], deq[0], torch.bfloat16)
        for config in (15, 16, 17) + ((18,) if blocks % 2 == 0 else ()):
            assert torch.equal(F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, torch.bfloat16, config=config).cpu(), want), (m, n, config)


@pytest.mark.parametrize("k", [256, 512, 765, 1021, 2048])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_split_tiles_on_both_sides_of_one_per_cu(dev, k, dtype):
    """256 and 272 split tiles (the two forms of the product), 2 to 16 k-blocks, the lean and the general epilogue, an addend, the swiglu form."""
    for m, n in ((1009, 4096), (1009, 4093), (1025, 4096), (1025, 4093)):
        F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, n, seed=k)
        want = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=16)
        assert torch.equal(F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=18), want), (m, n)
        if n % 32 == 0:
            add = torch.randn(m, n, device=dev).to(dtype)
            assert torch.equal(F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=18, addend=add),
                               F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=16, addend=add)), (m, n)
            assert torch.equal(F.bitlinear_mfma_swiglu(q[0], deq[0], qsum[0], pw, m, dtype), F.swiglu(want[:, :n // 2], want[:, n // 2:])), (m, n)


# the stream (410 rows) | split tiles: one per CU, two, three rounds | whole tiles: one per CU (15 k-blocks), four rounds; ragged rows and columns
@pytest.mark.parametrize("m,k,inter", [(410, 1024, 2816), (1009, 2048, 2016), (3833, 2048, 992), (2050, 1024, 2816), (2033, 1920, 2016), (5001, 1024, 2816)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_kernel_picked_for_the_swiglu_gives_the_same_bits(dev, m, k, inter, dtype):
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, 2 * inter, seed=3)
    y = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype, config=16)
    assert torch.equal(F.bitlinear_mfma_swiglu(q[0], deq[0], qsum[0], pw, m, dtype), F.swiglu(y[:, :inter], y[:, inter:]))


def test_odd_number_of_k_blocks_is_refused(dev):
    F, lib, pw, q, codes, deq, qsum = operands(dev, 70, 384, 256)
    with pytest.raises(RuntimeError):
        F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, 70, torch.bfloat16, config=18)


@pytest.mark.parametrize("m,k,inter", [(300, 2048, 1056), (333, 1024, 2816), (385, 1024, 2816), (66, 8448, 96)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_swiglu_equals_contraction_then_swiglu(dev, m, k, inter, dtype):
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, 2 * inter, seed=2)
    y = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, dtype)
    assert torch.equal(F.bitlinear_mfma_swiglu(q[0], deq[0], qsum[0], pw, m, dtype), F.swiglu(y[:, :inter], y[:, inter:]))


@pytest.mark.parametrize("seg", [512, 160])
def test_segments_contract_their_own_codes(dev, seg):
    m, k = 300, 512
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, 3 * seg, sets=3, seed=3)
    pw.wdeq, pw.seg_rows = pw.wdeq.repeat(3) * torch.tensor([1.0, 2.0, 0.5], device=dev), seg
    out = torch.empty(m, 3 * seg, dtype=torch.bfloat16, device=dev)
    F.L.check(lib.mmf_bitlinear_mfma_multi(q.data_ptr(), q.stride(0), deq.data_ptr(), qsum.data_ptr(), pw.packed.data_ptr(),
                                           pw.wdeq.data_ptr(), seg, out.data_ptr(), 3 * seg, m, k, 3 * seg, 1, 18, F.L.stream()), "multi")
    for s in range(3):
        alone = F.bitlinear_mfma(q[s], deq[s], qsum[s], pw, m, torch.bfloat16, config=5)
        assert torch.equal(out[:, s * seg:(s + 1) * seg], alone[:, s * seg:(s + 1) * seg]), s


@pytest.mark.parametrize("m,k,n", [(3968, 2048, 2048), (4147, 2048, 2048), (6387, 2048, 2048), (1216, 1792, 7168), (1216, 1536, 7168),
                                   (8256, 8704, 2048)])
def test_the_kernel_picked_beyond_one_round_of_split_tiles_gives_the_same_bits(dev, m, k, n):
    """496, 520 and 800 split tiles (two, three and four rounds of 256), 14 and 12 k-blocks at three rounds, five rounds of long rows."""
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, n, seed=4)
    picked = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, torch.bfloat16)
    for config in (16, 17, 18):
        assert torch.equal(picked, F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, torch.bfloat16, config=config)), config


@pytest.mark.parametrize("n", [4160, 4104, 4101])
@pytest.mark.parametrize("config", [15, 16, 17, 18])
def test_outputs_written_past_the_caches_are_the_same(dev, n, config):
    """2600 rows of bf16 outputs (21 MB) against their first 1312 alone (11 MB, the ordinary stores), ragged rows and columns, with an addend; one
    whose rows share lines, and a width that takes the general epilogue either way."""
    m, part, k = 2600, 1312, 256
    F, lib, pw, q, codes, deq, qsum = operands(dev, m, k, n, seed=5)
    add = torch.randn(m, n, device=dev).bfloat16()
    for kw in ({}, {"addend": add}):
        whole = F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, torch.bfloat16, config=config, **kw)
        first = {key: v[:part].contiguous() for key, v in kw.items()}
        assert torch.equal(whole[:part], F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, part, torch.bfloat16, config=config, **first))
        assert torch.equal(whole, F.bitlinear_mfma(q[0], deq[0], qsum[0], pw, m, torch.bfloat16, config=5, **kw))
