"""Forwards whose in-projection is written with a line between the channels (M a multiple of 8192 at d = 768): the bits of the dense
form, and modules of a caller's own see the dense form."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _encoder(gpu, L):
    import m2_amd
    cfg = m2_amd.m2_bert_80m(L)
    cfg.num_hidden_layers = 2
    enc = m2_amd.BertModel(cfg)
    enc.load_state_dict(m2_amd.seeded_state_dict(cfg, 3))
    return enc.encoder.to(gpu).eval()


class _Other(torch.nn.Module):
    """What a layer asks of an attention module, and nothing else."""

    def __init__(self, inner):
        super().__init__()
        self.inner, self.d_model = inner, inner.d_model
        self.residual_long_conv, self.hyena_training_additions = inner.residual_long_conv, False

    def project_in(self, x):
        return self.inner.project_in(x)

    def core(self, xproj, u_cm, B, L, spec=None):
        assert xproj.shape == (3 * self.d_model, B, L) and xproj.is_contiguous()
        return self.inner.core(xproj, u_cm, B, L, spec=spec)

    def project_out(self, y):
        return self.inner.project_out(y)


@pytest.mark.parametrize("L,B", [(256, 32), (512, 32)])
def test_rows_a_line_apart(gpu, L, B, monkeypatch):
    import m2_amd
    from m2_amd import ops
    enc, d, M = _encoder(gpu, L), 768, B * L
    assert ops.channels_row(M, d) > M
    h = torch.randn(B, L, d, generator=torch.Generator().manual_seed(B)).to(gpu)
    got = enc(h)[-1]
    enc.native_schedule = False
    seen = []
    real = ops.mixer_core
    monkeypatch.setattr(ops, "mixer_core", lambda x, *a, **kw: (seen.append(tuple(x.shape)), real(x, *a, **kw))[1])
    eager = enc(h)[-1]
    assert seen == [(3 * d, ops.channels_row(M, d))] * 2
    for i, at in enumerate(l.attention for l in enc.layer):      # a subclass, a core and a projection put in place of the module's
        if i == 0:
            at.core = lambda x, *a, at=at, **kw: m2_amd.MonarchMixerSequenceMixing.core(at, x, *a, **kw)
        else:
            at.project_in = lambda x, at=at: m2_amd.MonarchMixerSequenceMixing.project_in(at, x)
    seen.clear()
    replaced = enc(h)[-1]
    assert seen == [(3 * d, B, L)] * 2
    for at in (l.attention for l in enc.layer):
        at.__dict__.pop("core", None), at.__dict__.pop("project_in", None)
        at.__class__ = type("Own", (m2_amd.MonarchMixerSequenceMixing,), {})
    seen.clear()
    own = enc(h)[-1]
    assert seen == [(3 * d, B, L)] * 2
    assert all(torch.equal(eager, o) for o in (got, replaced, own))


def test_layer_with_an_attention_module_of_another_class(gpu):
    layer = _encoder(gpu, 256).layer[0]
    M, d = 8192, 768
    h = torch.randn(M, d, generator=torch.Generator().manual_seed(1)).to(gpu)
    args = h.bfloat16(), h.t().contiguous(), 32, 256, True
    with torch.no_grad():
        want = layer.fused(*args)[0]
        layer.attention = _Other(layer.attention)
        assert torch.equal(layer.fused(*args)[0], want)


@pytest.mark.parametrize("M,own", [(49152, True), (49280, False), (57344, False)])
def test_projections_of_very_many_rows(gpu, M, own):
    """On either side of the line beyond which the library's product takes over; a row a line apart is asked for on both."""
    import m2_amd
    from m2_amd import ops
    assert ops.own_to_channels(M, 768) == own
    g = torch.Generator(device=gpu).manual_seed(M)
    mixer = m2_amd.MonarchMixerSequenceMixing(768, l_max=128, hyena_filter_order=128, hyena_emb_dim=5).to(gpu)
    x = torch.randn(M, 768, generator=g, device=gpu).bfloat16()
    with torch.no_grad():
        got = mixer.projected(x, M // 128, 128).flatten(1)[:, :M]
    want = mixer.in_linear.weight.detach().bfloat16().float() @ x.float().t()
    assert (got.float() - want).norm() <= 2.0 ** -9 * want.norm() and (got.float() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
