"""Forwards of one or two sequences, whose mixer cores read filter taps, against the same ones on spectra: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _spectra_only(call):
    """The call with every core on spectra, and how many cores were on taps without that."""
    from m2_amd import ops, schedule  # noqa: F401
    kept, asked = ops.taps_pay, []
    ops.taps_pay = lambda B, L, dtype: (asked.append(kept(B, L, dtype)), False)[1]
    try:
        return call(), sum(asked)
    finally:
        ops.taps_pay = kept


@pytest.mark.parametrize("helper,L,residual,B", [("m2_bert_80m", 1024, True, 1), ("m2_bert_80m", 2048, False, 1), ("m2_bert_80m", 16384, True, 1),
                                                 ("m2_bert_110m", 4096, True, 1), ("m2_bert_large", 2048, True, 1), ("m2_bert_80m", 8192, True, 2)])
def test_few_sequences(gpu, helper, L, residual, B):
    import m2_amd
    cfg = getattr(m2_amd, helper)(L)
    cfg.num_hidden_layers, cfg.residual_long_conv = 2, residual
    model = m2_amd.BertModel(cfg)
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 3))
    model = model.to(gpu).eval()
    ids = torch.randint(0, cfg.vocab_size, (B, L), generator=torch.Generator().manual_seed(4)).to(gpu)
    with torch.no_grad():
        (want, pooled), taps = _spectra_only(lambda: model(ids))
        assert taps
        got, gpooled = model(ids)
        assert torch.equal(got, want) and torch.equal(gpooled, pooled)
        model.encoder.native_schedule = False
        for overlap in (None, False):
            model.encoder.overlap_filters = overlap
            assert torch.equal(model(ids)[0], got)
        model.encoder.overlap_filters = None
        layer = model.encoder.layer[0]
        u = torch.randn(B, L, cfg.hidden_size, generator=torch.Generator().manual_seed(5)).to(gpu).bfloat16()
        want, taps = _spectra_only(lambda: layer.attention(u)[0])
        assert taps == 1 and torch.equal(layer.attention(u)[0], want)


def test_mixers_of_a_callers_own_are_given_spectra(gpu):
    """A core put in the place of the module's, and kept spectra, see tensors as before; a graph of the taps route replays."""
    import m2_amd
    L = 1024
    cfg = m2_amd.m2_bert_80m(L)
    cfg.num_hidden_layers = 2
    model = m2_amd.BertModel(cfg, use_hip_graph=True)
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 6))
    model = model.to(gpu).eval()
    ids = [torch.randint(0, cfg.vocab_size, (1, L), generator=torch.Generator().manual_seed(s)).to(gpu) for s in (7, 8, 9)]
    with torch.no_grad():
        graphed = [model(i)[0] for i in ids]
        model.encoder.use_hip_graph = False
        assert all(torch.equal(model(i)[0], g) for i, g in zip(ids, graphed))
        model.encoder.native_schedule = False
        at, seen = model.encoder.layer[1].attention, []
        core = type(at).core

        def own(xproj, u, B, L, spec=None):
            seen.append(type(spec))
            return core(at, xproj, u, B, L, spec=spec)

        at.core = own
        assert torch.equal(model(ids[0])[0], graphed[0]) and seen == [torch.Tensor]
        del at.core
        at.cache_filters = True
        assert torch.equal(model(ids[0])[0], graphed[0]) and isinstance(at._spec_cache[1], torch.Tensor)


@pytest.mark.parametrize("L,B", [(1024, 1), (2048, 1), (4096, 2), (8192, 1), (16384, 1)])
def test_cached_filters_give_the_same_bits(gpu, L, B):
    """Kept spectra, spectra made layer by layer on the second stream and taps: three ways through the same forward."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(L)
    cfg.num_hidden_layers = 2
    model = m2_amd.BertModel(cfg)
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 10))
    model = model.to(gpu).eval()
    ids = torch.randint(0, cfg.vocab_size, (B, L), generator=torch.Generator().manual_seed(11)).to(gpu)
    with torch.no_grad():
        want = model(ids)[0]
        model.encoder.native_schedule = model.encoder.batch_filters = False
        for overlap in (True, "upfront"):
            model.encoder.overlap_filters = overlap
            assert torch.equal(model(ids)[0], want)
        for layer in model.encoder.layer:
            layer.attention.cache_filters = True
        assert all(torch.equal(model(ids)[0], want) for _ in range(2))


def test_a_second_input_without_a_second_filter(gpu):
    """`core` given an input for the residual convolution that the mixer does not have: as if it had not been given."""
    import m2_amd
    L, d = 1024, 768
    mixer = m2_amd.MonarchMixerSequenceMixing(d, l_max=L, bidirectional=True, hyena_emb_dim=5, hyena_filter_order=128, residual_long_conv=False,
                                              hyena_w=10).to(gpu).eval()
    g = torch.Generator().manual_seed(12)
    x, u = torch.randn(3 * d, 1, L, generator=g).to(gpu).bfloat16(), torch.randn(d, 1, L, generator=g).to(gpu)
    with torch.no_grad():
        y, z = mixer.core(x, u, 1, L), mixer.core(x, None, 1, L)
        assert torch.equal(y, z) and torch.equal(y, mixer.core(x, u, 1, L, spec=mixer.filter_spectrum(L)))
