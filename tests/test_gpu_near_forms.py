"""Activations rounded to 16 bits: the short evaluation with its fall-back gives the definition's bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_near_forms_give_the_definitions_bits(dev):
    """The bound on the near sigmoid for every float it is used on; every 16-bit argument, subnormals, infinities and NaNs among
    them, against 2048 values of the other operands (any magnitude, lower bounds outside [0, 1]) through each activation."""
    import matmulfreellm_amd._lib as L
    counts = torch.zeros(9, dtype=torch.int64, device=dev)
    with L.on(dev):
        L.check(L.load().mmf_diag_check_near_forms(2048, counts.data_ptr(), L.stream()), "mmf_diag_check_near_forms")
    print(f"near forms: outside the bound {counts[0]}, differing bf16 {counts[1:5].tolist()} fp16 {counts[5:].tolist()}", flush=True)
    assert counts.tolist() == [0] * 9


@pytest.mark.parametrize("k", [516, 1024, 2048, 2816])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_row_is_the_same_among_few_rows_and_many(dev, k, dtype):
    """Which evaluation a launch takes depends on its size (about 256 workgroups: 1024 or 2048 elements, or a row each); its bits do not."""
    import matmulfreellm_amd.functional as F
    torch.manual_seed(k)
    m = 1100
    x, a = torch.randn(m, k, device=dev).to(dtype) * 4, torch.randn(m, k, device=dev).to(dtype) * 4
    w, lb, state = (0.5 + torch.rand(k, device=dev)).to(dtype), torch.rand(k, device=dev), torch.randn(m, k, device=dev)
    def step(n):
        h = state[:n].clone()
        return [F.hgrn_step(x[:n], a[:n], h, lb), h]
    calls = {"swiglu": lambda n: [F.swiglu(x[:n], a[:n])], "swish gate": lambda n: [F.rmsnorm_swishgate(x[:n], a[:n], w)],
             "gate": lambda n: list(F.hgrn_gate(x[:n], a[:n], lb)), "step": step}
    for name, call in calls.items():
        whole = call(m)
        for n in (1, 85, 256, 257, 513):
            assert all(torch.equal(p, q[:n]) for p, q in zip(call(n), whole)), (name, n)
