"""The pooler as one kernel against fp64 and against the module, whose place it takes where that is plain."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [8, 264, 768, 960, 1536, 1792])
@pytest.mark.parametrize("B", [1, 2, 8, 9, 31, 256])
def test_against_fp64(gpu, B, d):
    from m2_amd import ops
    g = torch.Generator(device=gpu).manual_seed(B + d)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu)      # noqa: E731
    h, w, b = rn(B, 3, d), rn(d, d) / d ** 0.5, rn(d)
    h[0, 0, 0] = float("nan") if B > 1 else 1.0
    for bias in (b, None):
        got = ops.pooler(h[:, 0], w, bias)
        s = h[:, 0].double() @ w.double().t() + (0 if bias is None else bias.double())
        ref, size = s.tanh(), (h[:, 0].double().abs() @ w.double().abs().t() + 1)
        # sums of d products in fp32, in the root mean square far below d / 64 roundings of their size; tanh to two ulp
        bad = torch.isnan(ref)
        assert torch.equal(torch.isnan(got), bad)
        assert ((got.double() - ref).abs()[~bad] <= ((d / 64 + 8) * 2.0 ** -24 * size)[~bad]).all()


@pytest.fixture
def counted(gpu):
    """(a one-layer model, how often the kernel has run)"""
    import m2_amd
    from m2_amd import ops
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    model = m2_amd.BertModel(cfg)
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 2))
    calls, own = [], ops.pooler
    ops.pooler = lambda *a: (calls.append(1), own(*a))[1]
    yield model.to(gpu).eval(), calls
    ops.pooler = own


def _hidden(gpu, B=3):
    return torch.randn(B, 128, 768, generator=torch.Generator().manual_seed(B)).to(gpu)


def test_transforms_and_modes_see_the_module(gpu, counted):
    import torch.autograd.forward_ad as fw
    from torch.func import functional_call, jvp, vmap
    from torch.utils.flop_counter import FlopCounterMode
    model, calls = counted
    model.pooler.requires_grad_(False)
    h, p = _hidden(gpu), model.pooler
    w, dw = p.dense.weight.detach(), torch.randn_like(p.dense.weight)
    s = h[:, 0].double() @ w.double().t() + p.dense.bias.double()
    tangent = (h[:, 0].double() @ dw.double().t()) / s.cosh() ** 2

    class Pool(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.model = model

        def forward(self, h):
            return self.model._pool(h, None)

    m = Pool()
    assert torch.allclose(m(h).double(), s.tanh(), atol=1e-4) and len(calls) == 1
    with torch.device(gpu):                                       # (a default device is no such mode)
        m(h)
    assert len(calls) == 2
    name = "model.pooler.dense.weight"
    with fw.dual_level():
        out = fw.unpack_dual(functional_call(m, {name: fw.make_dual(w, dw)}, (h,)))
        assert torch.allclose(out.tangent.double(), tangent, atol=1e-3)
        out = fw.unpack_dual(m(fw.make_dual(h, torch.zeros_like(h))))
        assert out.tangent is not None
    out, t = jvp(lambda x: functional_call(m, {name: x}, (h,)), (w,), (dw,))
    assert torch.allclose(t.double(), tangent, atol=1e-3)
    many = vmap(lambda x: functional_call(m, {name: x}, (h,)))(torch.stack([w, 2 * w]))
    assert torch.allclose(many[0].double(), s.tanh(), atol=1e-4) and many.shape == (2, 3, 768)
    h.requires_grad_()
    assert m(h).requires_grad
    h.requires_grad_(False)
    with FlopCounterMode(display=False) as flops:
        m(h)
    assert flops.get_total_flops() == 2 * 3 * 768 * 768
    assert len(calls) == 2
    assert torch.jit.trace(m, (h,), check_trace=False)(2 * h).sub(torch.tanh(p.dense(2 * h[:, 0]))).abs().max() < 1e-5
    seen = []
    hook = torch.nn.modules.module.register_module_forward_hook(lambda mod, i, o: seen.append(mod))
    try:
        m(h)
    finally:
        hook.remove()
    assert p in seen and p.dense in seen and len(calls) == 2
    p.dense.compile()                                             # (is not run: only that it is asked for)
    p.dense._compiled_call_impl = lambda x: x + 1
    assert torch.equal(m(h), torch.tanh(h[:, 0] + 1)) and len(calls) == 2


def test_hidden_states_in_any_layout(gpu, counted):
    """What a caller's own encoder may return: the kernel takes rows it can read, the module everything else."""
    model, calls = counted
    h = _hidden(gpu, 5)
    with torch.no_grad():
        want = model.pooler(h)
        wide = torch.zeros(5, 128, 770, device=gpu)
        wide[..., :768] = h
        flat = torch.zeros(5 * (128 * 768 + 2), device=gpu)
        odd = flat.as_strided((5, 128, 768), (128 * 768 + 2, 768, 1))
        odd.copy_(h)
        shifted = torch.zeros(h.numel() + 1, device=gpu)[1:].view(h.shape)
        shifted.copy_(h)
        # (layout, sequences, whether the kernel takes it)
        for x, n, own in [(h, 5, True), (h.transpose(1, 2).contiguous().transpose(1, 2), 5, False), (wide[..., :768], 5, True),
                          (odd, 5, False), (odd[:1], 1, True), (shifted, 5, False), (h[:1].expand(5, 128, 768), 5, False), (h[::2], 3, True)]:
            del calls[:]
            got, ref = model._pool(x, None), model.pooler(x)
            assert len(calls) == own and got.shape == (n, 768) and (got - ref).abs().max() < 2e-6
        many = _hidden(gpu, 9)                                    # beyond what one pass over the weights serves
        del calls[:]
        assert torch.equal(model._pool(many, None), model.pooler(many)) and not calls
        assert model._pool(many[:8], None).shape == (8, 768) and len(calls) == 1
        assert model._pool(h[:0], None).shape == (0, 768) and (model._pool(h, None) - want).abs().max() < 2e-6
        with pytest.raises(IndexError):                           # no first token
            model._pool(h[:, :0], None)
        del calls[:]
        assert model.cpu()._pool(h.cpu(), None).device.type == "cpu" and not calls


def test_stands_for_the_module_only_where_it_is_plain(gpu):
    import m2_amd
    from m2_amd import ops
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    model = m2_amd.BertModel(cfg)
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 2))
    model = model.to(gpu).eval()
    ids = torch.randint(0, cfg.vocab_size, (3, 128), generator=torch.Generator().manual_seed(1)).to(gpu)
    calls, own = [], ops.pooler
    ops.pooler = lambda *a: (calls.append(1), own(*a))[1]
    try:
        with torch.no_grad():
            seq, pooled = model(ids)
            want = model.pooler(seq, mask=torch.ones_like(ids))
            assert len(calls) == 1 and (pooled - want).abs().max() < 1e-6
            with torch.autocast("cuda", dtype=torch.bfloat16):
                low = model(ids)[1]
            assert len(calls) == 1 and low.dtype == model.pooler.activation(torch.zeros(1, dtype=torch.bfloat16)).dtype
            hook = model.pooler.dense.register_forward_hook(lambda m, i, o: o + 1)
            assert (model(ids)[1] - (torch.atanh(want.double()) + 1).tanh()).abs().max() < 1e-4 and len(calls) == 1
            hook.remove()
        pooled = model(ids)[1]
        assert pooled.requires_grad and len(calls) == 1          # the module's own graph
        model.pooler.requires_grad_(False)
        assert not model(ids)[1].requires_grad and len(calls) == 2
    finally:
        ops.pooler = own
