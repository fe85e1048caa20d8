"""The calls that go from tensor to launch in native code: where they take over from the general path, and where they must not."""
import pytest
import torch

import matmulfreellm_amd as mm
import matmulfreellm_amd.functional as F
from matmulfreellm_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64,), (1, 64), (2, 4, 64), (8, 64), (9, 64), (0, 64), (3, 3, 64)])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, False), (torch.float32, False), (torch.float16, True)])
def test_few_rows_equal_the_general_path(dev, shape, dtype, bias):
    torch.manual_seed(0)
    layer = mm.FusedBitLinear(64, 40, bias=bias).to(dev, dtype)
    with torch.no_grad():
        layer.norm.weight.uniform_(0.5, 1.5)
        for x in (torch.randn(*shape, device=dev, dtype=dtype), torch.randn(*shape[:-1], 128, device=dev, dtype=dtype)[..., ::2],
                  torch.randn(torch.Size(shape).numel() + 1, device=dev, dtype=dtype)[1:].view(shape)):
            want = F.bitlinear(x.clone().view(-1, 64), layer.norm.weight, layer.packed_weight(), bias=layer.bias,
                               eps=layer.run_eps()).view(*shape[:-1], 40)
            if x.data_ptr() % 16 and x.is_contiguous() and x.numel():
                with pytest.raises(L.MMFError):
                    layer(x)
            else:
                assert torch.equal(layer(x), want)
        with pytest.raises(ValueError):
            layer(torch.randn(1, 65, device=dev, dtype=dtype))
        with pytest.raises(L.MMFError):
            layer(torch.randn(1, 64, dtype=dtype))
        one = torch.ones(1, 64, device=dev, dtype=dtype)
        before = layer(one)
        layer.weight.neg_()                                        # packed again when the weight is written
        assert bias or torch.equal(layer(one), -before)


@pytest.mark.parametrize("scan", [mm.fused_recurrent_hgrn, mm.chunk_hgrn])
@pytest.mark.parametrize("state,final", [(None, False), (torch.bfloat16, True)])
def test_native_scans_differentiate_like_autograd_of_the_recurrence(dev, scan, state, final):
    torch.manual_seed(1)
    b, h, t, d = 2, 3, 17, 40
    x = torch.randn(b, h, t, 2 * d, device=dev)[..., ::2].requires_grad_()
    gate = torch.sigmoid(torch.randn(b, t, h, d, device=dev)).transpose(1, 2)
    g = (gate.log() if scan is mm.chunk_hgrn else gate).requires_grad_()
    h0 = torch.randn(b, h, d, device=dev, dtype=state) if state else None
    o, last = scan(x, g, initial_state=h0, output_final_state=final)
    do = torch.randn_like(o)
    dx, dg = torch.autograd.grad(o, (x, g), do)
    x64, g64 = x.detach().double().requires_grad_(), g.detach().double().requires_grad_()
    s, out = h0.double() if state else torch.zeros(b, h, d, dtype=torch.double, device=dev), []
    for i in range(t):
        s = (g64[:, :, i].exp() if scan is mm.chunk_hgrn else g64[:, :, i]) * s + x64[:, :, i]
        out.append(s)
    ref = torch.stack(out, 2)
    rx, rg = torch.autograd.grad(ref, (x64, g64), do.double())
    for got, want in ((o, ref), (dx, rx), (dg, rg), *([(last, s)] if final else [])):
        assert torch.allclose(got.double(), want, rtol=1e-4, atol=1e-4)
    assert (last is None) != final and (last is None or (not last.requires_grad and last.dtype == torch.float32))
    with pytest.raises(ValueError):
        scan(x, g[:, :, :-1])
    with pytest.raises(L.MMFError):
        scan(x.detach().cpu().requires_grad_(), g)


def test_operands_of_another_size_are_refused(dev):
    """Per-column operands that are shorter or longer than the rows, gates of other sizes, layers of other widths: an error from the
    host, in every path, instead of a kernel that reads what is not there."""
    def refused(call, error=ValueError):
        with pytest.raises(error):
            call()

    w = lambda n, dtype=torch.float32: torch.ones(n, device=dev, dtype=dtype)
    for n in (32, 128):
        for x in (torch.randn(2, 64, device=dev), torch.randn(300, 64, device=dev)):
            layer = mm.FusedBitLinear(64, 40).to(dev)
            pw = layer.packed_weight()
            for grad in (False, True):
                with torch.set_grad_enabled(grad):
                    refused(lambda: mm.RMSNorm(n).to(dev)(x))
                    refused(lambda: mm.FusedRMSNormSwishGate(n).to(dev)(x, x))
                    other = mm.FusedBitLinear(64, 40).to(dev)
                    other.norm = mm.RMSNorm(n).to(dev)
                    refused(lambda: other(x))
                    biased = mm.FusedBitLinear(64, 40, bias=True).to(dev)
                    biased.bias = torch.nn.Parameter(w(n))
                    refused(lambda: biased(x))
            refused(lambda: F.bitlinear(x, w(64), pw, prologue=("norm", w(n), 1e-6)))
            refused(lambda: F.bitlinear(x, w(n), pw, prologue=("swiglu", x)))
            refused(lambda: F.rmsnorm_quant(x, w(n)))
    i = torch.zeros(3, 16, device=dev)
    for f in (torch.zeros(3, 8, device=dev), torch.zeros(2, 16, device=dev), torch.zeros(3, 16, device=dev, dtype=torch.bfloat16)):
        refused(lambda: F.hgrn_gate(i, f))
        refused(lambda: F.hgrn_step(i, f, torch.zeros(3, 16, device=dev)))
    refused(lambda: F.short_conv(torch.zeros(1, 5, 16, device=dev), torch.zeros(16, 1, 4, device=dev), w(8)))

    config = dict(vocab_size=100, hidden_size=64, num_hidden_layers=2, eos_token_id=None, bos_token_id=None)
    ids = torch.randint(0, 100, (1, 5), device=dev)
    for change in (lambda m: setattr(m.model.layers[1], "mlp", mm.HGRNBitMLP(64, intermediate_size=96).to(dev)),
                   lambda m: setattr(m, "lm_head", mm.FusedBitLinear(64, 80).to(dev)),
                   lambda m: setattr(m.model, "embeddings", torch.nn.Embedding(120, 64).to(dev))):
        model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(**config)).to(dev).eval()
        change(model)
        refused(lambda: model.generate(ids, max_new_tokens=3), NotImplementedError)
        assert model.generate(ids, max_new_tokens=3, use_graph=False).shape == (1, 8)
