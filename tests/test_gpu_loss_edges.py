"""The training loss at the edges of its passes over a row: one element, a row shorter than a pass, whole passes, remainders,
rows whose length or stride rules 16-byte accesses out -- against torch's loss in fp64 on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("v", [1, 7, 8, 511, 4096, 4104, 8193, 16384, 16392, 20001])
@pytest.mark.parametrize("pad", [0, 3])
def test_training_loss_row_edges(dev, dtype, v, pad):
    from matmulfreellm_amd.autograd import FusedCrossEntropyLoss
    torch.manual_seed(v)
    wide = (3 * torch.randn(3, v + pad)).to(dtype)
    labels = torch.tensor([0, v - 1, -100])
    ref = wide[:, :v].double().requires_grad_()
    want = torch.nn.functional.cross_entropy(ref, labels, reduction="sum")
    want.backward()
    got = wide.to(dev)[:, :v].requires_grad_()
    loss = FusedCrossEntropyLoss(reduction="sum")(got, labels.to(dev))
    loss.backward()
    assert abs(loss.item() - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    assert (got.grad.cpu().double() - ref.grad).abs().max().item() <= tol
