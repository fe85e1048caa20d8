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
