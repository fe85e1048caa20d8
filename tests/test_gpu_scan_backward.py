"""The scan backward at the edges of its split: block and segment remainders, halved columns (fewer than 256 of 64 channels),
whole columns, time segments with their carries, lanes past the last channel -- against autograd through the CPU
restatement, linear and log gates, with and without an initial state."""
import pytest
import torch

from oracle import hgrn as oh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("bhtd", [(1, 1, 1, 64), (1, 1, 24, 33), (1, 1, 25, 64), (1, 1, 48, 64), (1, 1, 49, 100), (1, 3, 431, 100),
                                  (1, 140, 50, 40), (1, 2, 23, 8200), (2, 1, 25, 8192), (1, 1, 2100, 96), (1, 2, 2497, 64)])
def test_scan_backward_split(dev, bhtd, log):
    import matmulfreellm_amd as mm
    torch.manual_seed(11)
    b, h, t, d = bhtd
    g = torch.randn(b, h, t, d) + 2
    g = torch.nn.functional.logsigmoid(g) if log else torch.sigmoid(g)
    x, do = torch.randn(b, h, t, d), torch.randn(b, h, t, d)
    h0 = torch.randn(b, h, d) if t % 2 else None
    leaves = [v.clone().requires_grad_() for v in (x, g)]
    o, _ = oh.naive_recurrent_hgrn_literal(leaves[0], leaves[1].exp() if log else leaves[1], h0, False)
    want = torch.autograd.grad(o, leaves, do)
    mine = [v.to(dev).requires_grad_() for v in (x, g)]
    o2, _ = (mm.chunk_hgrn if log else mm.fused_recurrent_hgrn)(*mine, h0.to(dev) if h0 is not None else None)
    got = torch.autograd.grad(o2, mine, do.to(dev))
    for name, a, r in zip(("dx", "dg"), got, want):
        err = ((a.cpu() - r).abs().max() / r.abs().max().clamp_min(1e-30)).item()
        assert err < 2e-5, (name, err)


@pytest.mark.parametrize("t", [64, 447, 448, 511, 512, 513])
@pytest.mark.parametrize("bh,d", [(1, 64), (63, 33), (64, 33)])
@pytest.mark.parametrize("chunk", [1, 7, 64])
def test_chunked_scan_where_the_time_axis_begins_to_be_cut(dev, t, bh, d, chunk):
    """Lengths on both sides of the first cut for every chunk length (448 is where two segments of four blocks fit, 8 blocks of
    whole chunks where a workspace is asked for) and of the number of columns above which nothing is cut; forward, final state
    and gradients against the sequential form in double precision.  An fp32 pass adds at most a few roundings per step to values
    that the gates damp: 2e-5 of the largest value, as the backward's bound above."""
    import matmulfreellm_amd as mm
    torch.manual_seed(t + bh)
    g = torch.nn.functional.logsigmoid(torch.randn(1, bh, t, d) + 2)
    x, do, h0 = torch.randn(1, bh, t, d), torch.randn(1, bh, t, d), torch.randn(1, bh, d)
    leaves = [v.double().requires_grad_() for v in (x, g)]
    h, steps = h0.double(), []
    for i in range(t):
        h = leaves[1][:, :, i].exp() * h + leaves[0][:, :, i]
        steps.append(h)
    want_o = torch.stack(steps, 2)
    want = [want_o, h, *torch.autograd.grad(want_o, leaves, do.double())]
    mine = [v.to(dev).requires_grad_() for v in (x, g)]
    o, last = mm.chunk_hgrn(*mine, h0.to(dev), output_final_state=True, chunk_size=chunk)
    got = [o, last, *torch.autograd.grad(o, mine, do.to(dev))]
    for name, a, r in zip(("o", "state", "dx", "dg"), got, want):
        err = ((a.detach().cpu().double() - r).abs().max() / r.abs().max()).item()
        assert err < 2e-5, (name, err)


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("bhtd", [(3, 5, 777, 96), (1, 2, 2497, 64), (2, 140, 300, 64)])
def test_scans_round_once_per_step(dev, bhtd, log):
    """Distance from 64 bits in fp32, gates sigmoid(N(1, 1)): an error of one unit roundoff (6e-8, rms 0.29 of it) per step, damped
    by the gates, comes to 3.7e-8 (backward, linear gates) and 4.5e-8 (log gates, with exp's own error) of the result's norm.  Two roundings a
    step, or the final rounding of l_t + P_t * carry on top of l_t's, give 5.3e-8 and 5.9e-8."""
    import matmulfreellm_amd as mm
    torch.manual_seed(3)
    x, do, z = (torch.randn(*bhtd, device=dev) for _ in range(3))
    g = (torch.nn.functional.logsigmoid if log else torch.sigmoid)(z + 1)
    xr, gr = x.clone().requires_grad_(), g.clone().requires_grad_()
    o, last = (mm.chunk_hgrn if log else mm.fused_recurrent_hgrn)(xr, gr, output_final_state=True)
    dx, _ = torch.autograd.grad(o, (xr, gr), do)
    a, h, dh = (g.double().exp() if log else g.double()), x.new_zeros(bhtd[0], bhtd[1], bhtd[3]).double(), 0.0
    hs, dhs = [], []
    for t in range(bhtd[2]):
        h = a[:, :, t] * h + x[:, :, t]
        hs.append(h)
    for t in reversed(range(bhtd[2])):
        dh = dh + do[:, :, t].double()
        dhs.append(dh)
        dh = dh * a[:, :, t]
    rel = lambda v, r: ((v.double() - r).norm() / r.norm()).item()
    assert rel(dx, torch.stack(dhs[::-1], 2)) < (5e-8 if log else 4.2e-8)
    assert rel(o, torch.stack(hs, 2)) < 5e-8
    assert rel(last, h) < 6e-8                       # as few as 128 values (their mean scatters by 5 %): one unit roundoff


@pytest.mark.parametrize("log", [False, True])
def test_a_zero_carry_survives_a_product_of_gates_that_overflows(dev, log):
    """40 gates of 1e4 (not a decay, but taken): their product is infinite, and what enters or leaves them is zero."""
    import matmulfreellm_amd as mm
    t = 200
    a = torch.full((1, 1, t, 64), 0.5)
    a[:, :, 60:100] = 1e4
    x, do = torch.zeros(1, 1, t, 64), torch.zeros(1, 1, t, 64)
    do[:, :, :50] = 1.0
    if not log:
        x[:, :, 150:] = 1.0
    g = a.log() if log else a
    mine = [v.to(dev).requires_grad_() for v in (x, g)]
    o, _ = (mm.chunk_hgrn if log else mm.fused_recurrent_hgrn)(*mine)
    dx, dg = torch.autograd.grad(o, mine, do.to(dev))
    want = torch.zeros(t)
    for k in reversed(range(50)):
        want[k] = 1.0 + 0.5 * want[k + 1]
    assert torch.isfinite(o).all() and torch.isfinite(dg).all()
    assert torch.allclose(dx[0, 0, :, 0].cpu(), want, rtol=1e-6, atol=0)


@pytest.mark.parametrize("bh,d,t", [(32, 64, 3072), (11, 130, 3101), (31, 64, 3072), (64, 64, 3100), (65, 33, 3073), (128, 64, 3361), (170, 40, 3080),
                                    (171, 40, 3080), (40, 64, 2050), (41, 64, 2050), (64, 64, 2050), (65, 64, 2050), (127, 33, 3071), (9, 512, 3072), (9, 512, 5121), (128, 32, 5120)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("log", [True, False])
def test_scans_whose_columns_are_shared_by_workgroups(dev, bh, d, t, dtype, log):
    """Long sequences around the numbers of columns (32, 64, 128, 170) and the lengths from which 8 to 3 workgroups take turns on one column or
    columns are halved: ragged columns, last rounds with fewer blocks than waves, an initial state; log gates and linear ones; twice, on the same
    buffers.  The bound is that of the cut sequences above; a 16-bit result is rounded once more (2^-8 of the value) and its gradients see a rounded o."""
    import matmulfreellm_amd as mm
    torch.manual_seed(bh + t)
    z = torch.randn(1, bh, t, d, device=dev) + 2
    g = (torch.nn.functional.logsigmoid if log else torch.sigmoid)(z).to(dtype)
    x, do, h0 = torch.randn(1, bh, t, d, device=dev).to(dtype), torch.randn(1, bh, t, d, device=dev).to(dtype), torch.randn(1, bh, d, device=dev)
    a, xd, dd = g[0].double().exp() if log else g[0].double(), x[0].double(), do[0].double()
    h, dh, hs, dhs = h0[0].double(), 0.0, [], []
    for i in range(t):
        h = a[:, i] * h + xd[:, i]
        hs.append(h)
    for i in reversed(range(t)):
        dh = dd[:, i] + dh
        dhs.append(dh)
        dh = dh * a[:, i]
    o = torch.stack(hs, 1)
    dx = torch.stack(dhs[::-1], 1)
    dg = dx * torch.cat([h0[0].double()[:, None], o[:, :-1]], 1)
    want = [o, h, dx, dg * a if log else dg]
    mine = [v.clone().requires_grad_() for v in (x, g)]
    for _ in range(2):
        got_o, last = (mm.chunk_hgrn if log else mm.fused_recurrent_hgrn)(*mine, h0, output_final_state=True)
        got = [got_o[0], last[0], *(v[0] for v in torch.autograd.grad(got_o, mine, do))]
        for name, p, r in zip(("o", "state", "dx", "dg"), got, want):
            err = ((p.detach().double() - r).abs().max() / r.abs().max()).item()
            assert err < (2e-5 if dtype == torch.float32 or name == "state" else 8e-3), (name, err)


def test_shared_columns_beside_other_streams(dev):
    """Three streams whose workgroups together are several times what the GPU holds, so that members of a column run without the others:
    every result is what the same call gives by itself, bit for bit (the carries are folded in one order, whoever does it)."""
    import matmulfreellm_amd as mm
    torch.manual_seed(5)
    calls = []
    for bh, t, d, dtype, log in ((128, 6000, 64, torch.bfloat16, True), (64, 9000, 64, torch.float32, False), (10, 5000, 1024, torch.float16, True)):
        z = torch.randn(1, bh, t, d, device=dev) + 1
        g = (torch.nn.functional.logsigmoid if log else torch.sigmoid)(z).to(dtype).requires_grad_()
        x, do = torch.randn(1, bh, t, d, device=dev).to(dtype).requires_grad_(), torch.randn(1, bh, t, d, device=dev).to(dtype)
        calls.append((mm.chunk_hgrn if log else mm.fused_recurrent_hgrn, x, g, do))
    def run(scan, x, g, do):
        o, last = scan(x, g, output_final_state=True)
        return [o.detach(), last, *torch.autograd.grad(o, (x, g), do)]
    alone = [run(*c) for c in calls]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in calls]
    together = [[] for _ in calls]
    for _ in range(4):
        for s, c, out in zip(streams, calls, together):
            with torch.cuda.stream(s):
                out.append(run(*c))
    torch.cuda.synchronize()
    for outs, want in zip(together, alone):
        for got in outs:
            assert all(torch.equal(a, b) for a, b in zip(got, want))


def _by_blocks(t, block, products, reverse, per_segment=None):
    """Gates of [t] steps whose products over the kernels' blocks (of 28 steps, backwards 24 from the last one on, counted anew in every
    `per_segment` of them) are `products` in turn, and 0.5 a step beyond."""
    a = torch.full((t,), 0.5, dtype=torch.double)
    per_segment = per_segment or -(-t // block)
    for s in range(0, t, per_segment * block):
        e = min(t, s + per_segment * block)
        blocks = [(i, min(e, i + block)) for i in range(s, e, block)]
        for (i, j), p in zip(blocks[::-1] if reverse else blocks, products):
            a[i:j] = p ** (1.0 / block)
    return a


@pytest.mark.parametrize("bh,per_segment,reverse,kind", [(32, None, r, k) for r in (False, True) for k in ("grows", "vanishes", "infinite")] +
                         [(1, 10, False, "grows"), (1, 11, True, "grows")])
def test_products_of_gates_keep_the_range_of_a_block(dev, bh, per_segment, reverse, kind):
    """Gates that are no decays, by blocks: columns shared by workgroups (32 of 3100 steps) and cut in time (one of 16384, 10 or 11 blocks a
    segment).  grows: a carry of 1e-25 passes blocks of 1e30, 1e30, 1e-30, 1e-30, whose product from the left overflows where the carry does not.
    vanishes: one of 1e-50 in front of 1e50: nothing is left of the carry, and no NaN.  infinite: an infinite carry stays infinite while
    each block's product is above zero."""
    import matmulfreellm_amd as mm
    t, block = 16384 if per_segment else 3100, 24 if reverse else 28
    products = {"grows": [1.0] * 2 + [1e30, 1e30, 1e-30, 1e-30] + [1.0] * 4, "vanishes": [1.0, 1e-50, 1e50] + [1.0] * 7, "infinite": []}[kind]
    if per_segment and kind == "grows":                # by waves: two blocks of 1e25 in one's hands, two of 1e-25 in another's
        products = [1e25, 1e-25] + [1.0] * 6 + [1e25, 1e-25, 1.0]
    a = _by_blocks(t, block, products, reverse, per_segment)
    g = a.float()[None, None, :, None].expand(1, bh, t, 64).contiguous()
    x, do, h0 = torch.zeros(1, bh, t, 64), torch.zeros(1, bh, t, 64), torch.zeros(1, bh, 64)
    start = {"grows": 1e-25, "vanishes": 1.0, "infinite": float("inf")}[kind]
    if reverse:
        do[:, :, -1] = start
    else:
        h0[:] = start
    mine = [v.to(dev).requires_grad_() for v in (x, g.double().log().float() if not reverse else g)]
    o, last = (mm.fused_recurrent_hgrn if reverse else mm.chunk_hgrn)(*mine, h0.to(dev), output_final_state=True)
    got = torch.autograd.grad(o, mine, do.to(dev))[0] if reverse else o.detach()
    gd = g[0, 0, :, 0].double()
    if reverse:
        want = start * torch.cat([gd.flip(0).cumprod(0).flip(0)[1:], torch.ones(1, dtype=torch.double)])
    else:
        want = start * gd.cumprod(0)
    got = got[0, :, :, ::9].double().cpu()
    if kind == "infinite":
        assert torch.isinf(got).all()
    elif kind == "vanishes":
        assert torch.isfinite(got).all()
    else:                                               # 28 roundings of a log gate of 2.5 a block, exp's own, and denormal ends
        assert ((got - want[None, :, None]).abs() <= 1e-4 * want[None, :, None] + 1e-37).all()


def test_workspace_of_shared_columns(dev):
    """The C entries: a workspace at any multiple of 4 bytes serves the same plan (same bits); none is an error where the sequence has to be cut, as
    for fewer than 128 columns it always had, and leaves it whole from there on."""
    from matmulfreellm_amd import _lib as L
    lib = L.load()
    torch.manual_seed(2)
    for bh, refused in ((32, True), (127, True), (128, False), (170, False)):
        t, d = 3100, 64
        x, do, z = (torch.randn(bh, t, d, device=dev) for _ in range(3))
        g = torch.nn.functional.logsigmoid(z + 1)
        nbytes = max(lib.mmf_hgrn_chunk_workspace_bytes(bh, t, d, 64), lib.mmf_hgrn_recurrent_bwd_workspace_bytes(bh, t, d))
        ws = torch.full((nbytes // 4 + 4,), float("nan"), device=dev)
        results = []
        for at in (0, 4):
            o, dx, dg = (torch.zeros_like(x) for _ in range(3))
            p = ws.data_ptr() + at
            L.check(lib.mmf_hgrn_chunk(x.data_ptr(), g.data_ptr(), None, o.data_ptr(), None, bh, t, d, 64, L.dtype_id(x.dtype), p, L.stream()), "fwd")
            L.check(lib.mmf_hgrn_recurrent_bwd_split(g.data_ptr(), o.data_ptr(), do.data_ptr(), None, dx.data_ptr(), dg.data_ptr(), bh, t, d, 1,
                                                     L.dtype_id(x.dtype), p, L.stream()), "bwd")
            results.append((o, dx, dg))
        assert all(torch.equal(a, b) for a, b in zip(*results))
        assert all(torch.isfinite(a).all() for a in results[0])
        o = torch.zeros_like(x)
        rc = lib.mmf_hgrn_chunk(x.data_ptr(), g.data_ptr(), None, o.data_ptr(), None, bh, t, d, 64, L.dtype_id(x.dtype), None, L.stream())
        assert (rc != 0) == refused
        if not refused:
            assert torch.allclose(o, results[0][0], rtol=1e-4, atol=1e-5)
