"""Decode with inner norms of their own behind i, f and g (a trained checkpoint): every path the engine has for a batch --
resident launch, one launch per BitLinear, quantiser + matrix cores, one launch per op -- gives the module path's logits
and states bit for bit.  Layers that agree and layers that differ in one model."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,dtype", [(512, torch.bfloat16), (2048, torch.float16), (160, torch.bfloat16), (96, torch.float32)])
@pytest.mark.parametrize("batch", [1, 5, 8, 9, 40])
def test_engine_steps_equal_module_steps(dev, hidden, dtype, batch):
    import matmulfreellm_amd as mm
    torch.manual_seed(17)
    model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=300, hidden_size=hidden, num_hidden_layers=3, eos_token_id=None))
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name and ".layers.1.attn" not in name:
                p.copy_(0.5 + torch.rand(p.shape))
            if name.endswith("lower_bounds"):
                p.copy_(torch.randn(p.shape))
    model = model.to(dev, dtype).eval()
    ids = torch.randint(0, 300, (batch, 7), device=dev)
    with torch.no_grad():
        out = model(input_ids=ids, use_cache=True, logits_to_keep=1)
        states = [s[-1].clone() for s in out.past_key_values]
        tok, want = out.logits[:, -1].argmax(-1), []
        for _ in range(3):
            out = model(input_ids=tok.view(-1, 1), past_key_values=out.past_key_values, use_cache=True)
            want.append(out.logits[:, -1].clone())
            tok = out.logits[:, -1].argmax(-1)
        first = model(input_ids=ids, use_cache=True, logits_to_keep=1).logits[:, -1].argmax(-1)
        paths = [(True, None), (False, None)] + ([(True, False)] if batch == 1 else [])
        for fuse, resident in paths:
            eng = mm.DecodeEngine(model, batch, fuse=fuse, resident=resident)
            if fuse and resident is None and batch == 1 and hidden % 128 == 0:
                assert eng.resident and eng.norms == 3
            eng.load_state(states)
            tok = first
            for w in want:
                logits = eng.step(tok)
                assert torch.equal(logits, w), (fuse, resident, eng.resident, eng.fused, eng.fused_mfma)
                tok = logits.argmax(-1)
            eng.check()
            for a, b in zip(eng.export_state(), (s[-1] for s in out.past_key_values)):
                assert torch.equal(a.view(-1), b.reshape(-1))


@pytest.mark.parametrize("hidden,layers,resident", [(4096, 5, True), (4096, 6, False), (2560, 20, False)])
def test_a_model_that_outgrows_the_resident_launch_decodes_through_the_launch_chain(dev, hidden, layers, resident):
    """Three inner norms behind i, f and g at the widest rows: the largest number of layers whose table and buffers fit the LDS of a
    CU, and the first that does not.  generate() and the engine work on both sides."""
    import matmulfreellm_amd as mm
    with torch.device("meta"):
        model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=300, hidden_size=hidden, num_hidden_layers=layers, eos_token_id=None,
                                                       intermediate_size=8192 if hidden == 4096 else None))
    model = model.to(torch.bfloat16).to_empty(device=dev).eval()
    gen = torch.Generator(device=dev).manual_seed(5)
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(0.5 + torch.rand(p.shape, generator=gen, device=dev) if "norm" in name
                    else torch.randn(p.shape, generator=gen, device=dev) * 0.02)
        ids = torch.randint(0, 300, (1, 9), generator=gen, device=dev)
        out = model(input_ids=ids, use_cache=True, logits_to_keep=1)
        toks = [out.logits[:, -1].argmax(-1)]
        for _ in range(4):
            out = model(input_ids=toks[-1].view(1, 1), past_key_values=out.past_key_values, use_cache=True)
            toks.append(out.logits[:, -1].argmax(-1))
        assert torch.equal(model.generate(ids, max_new_tokens=5)[0, 9:], torch.cat(toks))
        eng = mm.DecodeEngine.for_model(model, 1)
        assert eng.norms == 3 and eng.fused and eng.resident == resident
        assert torch.equal(eng.logits, out.logits[:, -1])
        for a, b in zip(eng.export_state(), (s[-1] for s in out.past_key_values)):
            assert torch.equal(a.view(-1), b.reshape(-1))
        if not resident:
            with pytest.raises(mm._lib.MMFError):
                mm.DecodeEngine(model, 1, resident=True)
