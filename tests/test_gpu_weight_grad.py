"""Weight gradients, several products of one launch: dout^T @ y in fp32 sums."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# rows: one stage and less, its edges, the buffers' edges, rows cut into slices; outputs: tiles' edges, several tiles and panels
CASES = [(1, [(8, 8)]), (31, [(256, 256)]), (32, [(248, 264), (8, 512)]), (33, [(256, 256)]), (95, [(264, 520)]), (128, [(512, 256)]),
         (129, [(264, 1304), (40, 16)]), (161, [(256, 1288)]), (1056, [(1024, 1024), (264, 72)]), (2017, [(2048, 2048)] * 4 + [(520, 264)]),
         (4099, [(256, 256)] * 8)]


def grads(pairs, dtype):
    from matmulfreellm_amd import _lib as L
    lib = L.load()
    p, q, m = ctypes.c_void_p * len(pairs), ctypes.c_int64 * len(pairs), pairs[0][0].shape[0]
    out = [torch.full((d.shape[1], y.shape[1]), float("nan"), dtype=dtype, device=d.device) for d, y in pairs]
    ns, ks = q(*[d.shape[1] for d, _ in pairs]), q(*[y.shape[1] for _, y in pairs])
    size = lib.mmf_weight_grad_workspace_bytes(len(pairs), ns, ks, m, L.dtype_id(dtype))
    ws = torch.empty(max(size, 1), dtype=torch.uint8, device=out[0].device)
    rc = lib.mmf_weight_grad(len(pairs), p(*[d.data_ptr() for d, _ in pairs]), q(*[d.stride(0) for d, _ in pairs]),
                             p(*[y.data_ptr() for _, y in pairs]), q(*[y.stride(0) for _, y in pairs]), p(*[o.data_ptr() for o in out]),
                             ns, ks, m, L.dtype_id(dtype), ws.data_ptr(), L.stream())
    return rc, out, size


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,shapes", CASES)
def test_weight_gradients_are_the_products(dev, m, shapes, dtype):
    """Within half a unit of the rounding and m of the sums'; strided gradients; rows and columns around the operands must not join."""
    g = torch.Generator().manual_seed(m)
    pairs = []
    for n, k in shapes:
        d = torch.full((m + 1, n + 16), float("nan"), dtype=dtype)
        y = torch.full((m + 1, k + 8), float("inf"), dtype=dtype)
        d[:m, 8:8 + n], y[:m, :k] = torch.randn(m, n, generator=g).to(dtype), torch.randn(m, k, generator=g).to(dtype)
        pairs.append((d.to(dev)[:m, 8:8 + n], y.to(dev)[:m, :k]))
    rc, out, size = grads(pairs, dtype)
    assert rc == 0 and (m not in (1056, 2017, 4099) or size > 0 or dtype == torch.float32)
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
    for (d, y), o in zip(pairs, out):
        want, scale = d.double().t() @ y.double(), d.double().abs().t() @ y.double().abs()
        # fp16 results below 2^-14 round to a multiple of 2^-24
        assert bool(((o.double() - want).abs() <= eps * want.abs() + m * 2.0 ** -24 * scale + 2.0 ** -25).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,shapes", [c for c in CASES if c[0] > 161])
def test_many_rows_lose_no_bits_of_their_operands(dev, m, shapes, dtype):
    """Sums of at most nine terms that are not zero, rows m // 8 apart: within half a unit of the rounding and nine of the sums', where m units of a full sum
    would hide operands of 11 bits."""
    g = torch.Generator().manual_seed(m)
    apart = m // 8
    pairs = []
    for n, k in shapes:
        y = torch.randn(m, k, generator=g) * (torch.arange(m)[:, None] % apart == torch.arange(k) % apart)
        pairs.append((torch.randn(m, n, generator=g).to(dtype).to(dev), y.to(dtype).to(dev)))
    rc, out, _ = grads(pairs, dtype)
    assert rc == 0
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
    for (d, y), o in zip(pairs, out):
        want, scale = d.double().t() @ y.double(), d.double().abs().t() @ y.double().abs()
        assert bool(((o.double() - want).abs() <= eps * want.abs() + 9 * 2.0 ** -24 * scale + 2.0 ** -25).all())


def test_not_a_number_reaches_its_row_and_column_only(dev):
    d, y = torch.ones(70, 264, dtype=torch.bfloat16, device=dev), torch.ones(70, 272, dtype=torch.bfloat16, device=dev)
    d[69, 263], y[3, 270] = float("nan"), float("inf")
    rc, (o,), _ = grads([(d, y)], torch.bfloat16)
    assert rc == 0 and bool(o[263].isnan().all()) and bool((o[:263, 270] == float("inf")).all())
    o[263], o[:, 270] = 70, 70
    assert bool((o == 70).all())


def test_weight_gradients_refuse_what_they_do_not_read(dev):
    from matmulfreellm_amd import _lib as L
    d, y = torch.ones(64, 264, dtype=torch.bfloat16, device=dev), torch.ones(64, 256, dtype=torch.bfloat16, device=dev)
    assert grads([(d[:, :260], y)], torch.bfloat16)[0] == -3
    assert grads([(d[:, 4:260], y)], torch.bfloat16)[0] == -3
    assert grads([(d, y)] * 9, torch.bfloat16)[0] == -1
    assert grads([(d.float()[:, :262], y.float())], torch.float32)[0] == -3
