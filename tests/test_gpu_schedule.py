"""The native schedule of an encoder (m2_amd/schedule.py) against the Python schedule: the same bits in every form, and plans
that follow their modules."""
import copy
import weakref

import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(cfg, gpu, seed, **kw):
    import m2_amd
    model = m2_amd.BertModel(cfg, **kw)
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, seed))
    return model.to(gpu).eval()


def _counted(call):
    """(result, how often a plan ran for it)"""
    from m2_amd import schedule
    run, calls = schedule.StackPlan.run, []

    def counting(self, *args, **kw):
        calls.append(self)
        return run(self, *args, **kw)

    schedule.StackPlan.run = counting
    try:
        return call(), len(calls)
    finally:
        schedule.StackPlan.run = run


def _both(model, *args, encoder_only=False, **kw):
    """(native result, Python-schedule result); a plan must have run for the first and none for the second."""
    call = model.encoder if encoder_only else model
    model.encoder.native_schedule = True
    got, runs = _counted(lambda: call(*args, **kw))
    model.encoder.native_schedule = False
    want, none = _counted(lambda: call(*args, **kw))
    model.encoder.native_schedule = True
    assert (runs, none) == (1, 0)
    return got, want


def _ids(cfg, B, L, seed, gpu):
    return torch.randint(0, cfg.vocab_size, (B, L), generator=torch.Generator().manual_seed(seed)).to(gpu)


# few rows, one-kernel MLP, streaming GLU with and without few rows, l_max beyond L
@pytest.mark.parametrize("helper,l_max,B,L", [("m2_bert_80m", 128, 1, 128), ("m2_bert_80m", 512, 3, 512), ("m2_bert_80m", 1024, 5, 256),
                                              ("m2_bert_110m", 128, 1, 128), ("m2_bert_large", 256, 3, 256), ("m2_bert_341m", 128, 2, 128)])
def test_native_schedule_matches_python_schedule(gpu, helper, l_max, B, L):
    import m2_amd
    cfg = getattr(m2_amd, helper)(l_max)
    cfg.num_hidden_layers = 3
    model = _model(cfg, gpu, 5)
    ids = _ids(cfg, B, L, 6, gpu)
    mask = torch.ones_like(ids)
    (seq, pooled), (wseq, wpooled) = _both(model, ids, attention_mask=mask)
    assert torch.equal(seq, wseq) and torch.equal(pooled, wpooled)
    (all_, _), (wall, _) = _both(model, ids, output_all_encoded_layers=True)
    assert len(all_) == 3 and all(torch.equal(a, b) for a, b in zip(all_, wall))
    tt = (ids % 2).contiguous()
    pos = torch.arange(L, device=gpu).flip(0)[None]
    (a, _), (b, _) = _both(model, ids, token_type_ids=tt, position_ids=pos)
    assert torch.equal(a, b) and not torch.equal(a, seq)
    h = torch.randn(B, L, cfg.hidden_size, generator=torch.Generator().manual_seed(7)).to(gpu)
    outs, want = _both(model, h, encoder_only=True)
    assert len(outs) == 3 and all(torch.equal(a, b) for a, b in zip(outs, want))


def test_plans_follow_their_modules(gpu):
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 2
    model = _model(cfg, gpu, 8)
    ids = _ids(cfg, 2, 128, 9, gpu)
    (prev, _), _ = _both(model, ids)
    lay = model.encoder.layer[1]

    def changed(what):
        nonlocal prev
        (got, _), (want, _) = _both(model, ids)
        assert torch.equal(got, want) and not torch.equal(got, prev), what
        prev = got

    with torch.no_grad():
        lay.attention.out_linear.weight.mul_(1.5)                              # in place: a copy has to be made again
        changed("weight in place")
        lay.mlp.wo.bias.add_(0.5)                                              # read in place
        changed("bias in place")
        lay.attention.filter_fn.implicit_filter[6].weight.mul_(2.0)
        changed("filter in place")
        lay.mlp.gated_layers.weight = torch.nn.Parameter(lay.mlp.gated_layers.weight.detach() * 1.2)
        changed("parameter replaced")
        lay.attention.in_linear.weight.data = lay.attention.in_linear.weight.data * 1.1
        changed("data replaced")
    new = torch.nn.LayerNorm(768, eps=cfg.layer_norm_eps).to(gpu)
    torch.nn.init.constant_(new.weight, 0.7)
    lay.mlp.layernorm = new
    changed("module replaced")
    model.embeddings.word_embeddings = torch.nn.Embedding.from_pretrained(model.embeddings.word_embeddings.weight.detach() * 0.5)
    changed("embedding replaced")
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 10))
    changed("state dict loaded")
    model.encoder.layer.append(copy.deepcopy(lay))                             # one more layer
    changed("layer added")
    fresh = _model(cfg, gpu, 10)
    want, _ = fresh(ids)
    got, _ = copy.deepcopy(fresh)(ids)                                         # a copy makes plans of its own
    assert torch.equal(got, want)
    lay.mlp.bf16_presum = False                                                # an option the native schedule has no path for
    opt, _ = model(ids)
    assert not torch.equal(opt, prev)


def test_native_schedule_in_a_graph_and_on_streams(gpu):
    """Captured and replayed with other work in between; eager calls on two streams at once."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(256)
    cfg.num_hidden_layers = 2
    model, graphed = _model(cfg, gpu, 11), _model(cfg, gpu, 11, use_hip_graph=True)
    for it in range(4):
        ids = _ids(cfg, 3, 256, 20 + it, gpu)
        want, _ = model(ids)
        scratch = torch.randn(512, 512, device=gpu) @ torch.randn(512, 512, device=gpu)
        got, _ = graphed(ids)
        torch.cuda.synchronize()
        assert torch.equal(got, want), it
        del scratch
    model.validate_ids = False
    batches = [_ids(cfg, 3, 256, 30 + i, gpu) for i in range(6)]
    wants = [model(b)[0].clone() for b in batches]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = []
    for i, b in enumerate(batches):
        with torch.cuda.stream(streams[i % 2]):
            outs.append(model(b)[0])
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(outs, wants))


def test_bad_indices_are_reported_by_the_native_schedule(gpu):
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    model = _model(cfg, gpu, 12)
    ids = _ids(cfg, 1, 128, 13, gpu)
    model(ids)
    assert model.encoder._native_plans
    ids[0, 5] = cfg.vocab_size
    with pytest.raises(IndexError):
        model(ids)
    ids[0, 5] = 0
    model(ids)


def test_a_graph_keeps_what_it_reads(gpu):
    """Forwards of other lengths replace the pointer tables of plans and schedules: a captured graph holds on to its own."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(512)
    cfg.num_hidden_layers = 1
    for native in (True, False):
        model = _model(cfg, gpu, 14, use_hip_graph=True)
        model.encoder.native_schedule = native
        ids = _ids(cfg, 2, 128, 15, gpu)
        first, _ = model(ids)
        table = next(iter(model.encoder._native_plans.values())).table if native else model.encoder._filter_table[1]
        held, address = table.table, table.table.data_ptr()
        gone = weakref.ref(table)
        del table, held
        model.encoder._native_plans.clear()
        model.encoder._filter_table = None
        for L in (256, 512):
            model(_ids(cfg, 2, L, L, gpu))
        assert gone() is not None and gone().table.data_ptr() == address
        again, _ = model(ids)
        assert torch.equal(again, first)
        model.encoder.reset_graphs()
        model.encoder._native_plans.clear()
        model.encoder._filter_table = None
        assert gone() is None


@pytest.mark.parametrize("native", [True, False])
def test_an_input_that_requires_grad_is_refused(gpu, native):
    """There is no backward: hidden states that require grad raise instead of coming back detached."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    enc = m2_amd.BertEncoder(cfg).to(gpu).eval()
    enc.native_schedule = native
    h = torch.randn(2, 128, 768, generator=torch.Generator().manual_seed(1)).to(gpu)
    want = enc(h)[-1]
    h.requires_grad_()
    with pytest.raises(RuntimeError):
        enc(h)
    with torch.no_grad():
        assert torch.equal(enc(h)[-1], want)


def test_a_weight_at_the_address_of_an_earlier_one(gpu):
    """Plans outlive weights that are replaced while forwards of another length run; an address comes back (as the allocator
    gives it out again) and `.data` keeps the version counter: the plan must not take the new weight for the old one."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(256)
    cfg.num_hidden_layers = 1
    model = _model(cfg, gpu, 21)
    short, long = _ids(cfg, 1, 128, 22, gpu), _ids(cfg, 1, 256, 23, gpu)
    at, mlp = model.encoder.layer[0].attention, model.encoder.layer[0].mlp
    for lin in (at.in_linear, at.out_linear, mlp.gated_layers, mlp.wo):
        memory = lin.weight.detach().clone()
        lin.weight.data = torch.from_dlpack(memory)             # a storage of its own on that memory
        (before, _), _ = _both(model, short)
        address, version = lin.weight.data_ptr(), lin.weight._version
        lin.weight.data = memory * 1.5
        model(long)                                             # the module's own copy is made anew here
        memory.mul_(2.0)
        lin.weight.data = torch.from_dlpack(memory)
        assert (lin.weight.data_ptr(), lin.weight._version) == (address, version)
        (got, _), (want, _) = _both(model, short)
        assert torch.equal(got, want) and not torch.equal(got, before)


def test_plans_follow_plain_values(gpu):
    """Epsilons, filter constants and options are read by every forward: a plan made before they were changed is not used."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 2
    model = _model(cfg, gpu, 24)
    ids = _ids(cfg, 2, 128, 25, gpu)
    (prev, _), _ = _both(model, ids)
    lays = model.encoder.layer

    def changed(what):
        nonlocal prev
        model.encoder.native_schedule = True
        (got, _), runs = _counted(lambda: model(ids))
        assert runs == (0 if what == "one layer's epsilon" else 1), what        # (layers that differ: the Python schedule)
        model.encoder.native_schedule = False
        want, _ = model(ids)
        assert torch.equal(got, want) and not torch.equal(got, prev), what
        prev = got

    lays[1].mlp.layernorm.eps = 0.3
    changed("one layer's epsilon")
    lays[0].mlp.layernorm.eps = 0.3
    changed("both layers' epsilon")
    model.embeddings.LayerNorm.eps = 0.2
    changed("epsilon of the embeddings")
    for lay in lays:
        for f in (lay.attention.filter_fn, lay.attention.filter_fn2):
            f.modulation.shift = 0.1
    changed("shift")
    for lay in lays:
        for f in (lay.attention.filter_fn, lay.attention.filter_fn2):
            f.w_mod = 2
    changed("w_mod")
    for lay in lays:
        lay.attention.residual_long_conv = False
    changed("without the residual convolution")
    model.embeddings.use_positional_encodings = False
    changed("without positions")


def test_a_narrowed_table_and_wrong_shapes(gpu):
    """Rows cut off a table after a plan was made are rows no id may name; a parameter of another shape is refused, not read past its
    end."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    model = _model(cfg, gpu, 26)
    ids = _ids(cfg, 1, 128, 27, gpu) % 1000
    ids[0, 3] = 2000
    before, _ = model(ids)
    word = model.embeddings.word_embeddings
    word.weight.data = word.weight.data[:1000]
    with pytest.raises(IndexError):
        model(ids)
    ids[0, 3] = 999
    (got, _), (want, _) = _both(model, ids)
    assert torch.equal(got, want)
    mlp, at = model.encoder.layer[0].mlp, model.encoder.layer[0].attention
    for mod, key, shape in ((mlp.layernorm, "weight", (512,)), (mlp.layernorm, "bias", (512,)), (mlp.wo, "bias", (700,)),
                            (at.in_linear, "weight", (2304, 512)), (at.out_linear, "weight", (512, 768)), (at.short_filter, "bias", (768,))):
        was = mod._parameters[key]
        mod._parameters[key] = torch.nn.Parameter(torch.zeros(shape, device=gpu))
        with pytest.raises((ValueError, RuntimeError)):
            model(ids)
        mod._parameters[key] = was
    again, _ = model(ids)
    assert torch.equal(again, got)


def test_computed_weights_and_other_classes_take_the_python_schedule(gpu):
    """Parametrised, weight-normed and pruned weights, subclasses and modules without a plan's parameters: a forward runs as with
    the native schedule off."""
    import m2_amd
    from m2_amd import encoder as enc, mixer
    from torch.nn.utils import parametrize, prune
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 2
    ids = _ids(cfg, 1, 128, 28, gpu)

    class Halved(torch.nn.Module):
        def forward(self, w):
            return w * 0.5

    class OwnLayer(enc.BertLayer):
        def fused(self, *args, **kw):
            o32, h16, hT = super().fused(*args, **kw)
            return None if o32 is None else o32 + 1, h16, hT

    class OwnMixer(mixer.MonarchMixerSequenceMixing):
        def project_out(self, y, *args):
            return super().project_out(y, *args) * 2

    class OwnMLP(enc.BertGatedLinearUnitMLP):
        def normed(self, a16, *args):
            return super().normed(a16 * 2, *args)

    class OwnLinear(m2_amd.BlockdiagLinear):
        def weight_bf16(self):
            return super().weight_bf16() * 2

    def retype(mod, cls):
        mod.__class__ = cls

    changes = {
        "parametrised": lambda lay: parametrize.register_parametrization(lay.attention.in_linear, "weight", Halved()),
        "block-diagonal parametrised": lambda lay: parametrize.register_parametrization(lay.mlp.wo, "weight", Halved()),
        "filter parametrised": lambda lay: parametrize.register_parametrization(lay.attention.filter_fn.implicit_filter[4], "weight", Halved()),
        "weight norm": lambda lay: torch.nn.utils.parametrizations.weight_norm(lay.attention.out_linear),
        "pruned": lambda lay: prune.random_unstructured(lay.attention.out_linear, "weight", 0.5),
        "layer": lambda lay: retype(lay, OwnLayer), "mixer": lambda lay: retype(lay.attention, OwnMixer),
        "option": lambda lay: setattr(lay.mlp, "bf16_presum", False), "mlp": lambda lay: retype(lay.mlp, OwnMLP), "linear": lambda lay: retype(lay.mlp.gated_layers, OwnLinear)}
    for what, change in changes.items():
        for first in (False, True):                  # changed before any plan, and after one was made
            model = _model(cfg, gpu, 29)
            before, _ = model(ids)
            if first:
                model.encoder._native_plans.clear()
            torch.manual_seed(1)
            change(model.encoder.layer[1])
            (got, _), runs = _counted(lambda: model(ids))
            assert runs == 0, what
            model.encoder.native_schedule = False
            want, _ = model(ids)
            assert torch.equal(got, want), what
            if what != "weight norm":                # (that one keeps the values)
                assert not torch.equal(got, before), what
            model.encoder.native_schedule = True     # that there is no plan is remembered, until something changes
            none = model.encoder._native_plans[128]
            assert torch.equal(model(ids)[0], want) and not none.usable and model.encoder._native_plans[128] is none, what
            model.encoder.layer[1] = _model(cfg, gpu, 29).encoder.layer[1]
            assert torch.equal(model(ids)[0], before) and model.encoder._native_plans[128].usable, what


def test_a_layer_class_with_the_plain_signature(gpu):
    import m2_amd
    from m2_amd import encoder as enc

    class Plain(enc.BertLayer):
        def fused(self, h16, hT, B, L, want_f32, spec=None, spec_ready=None, after_core=None, h32=None):
            return super().fused(h16, hT, B, L, want_f32, spec=spec, spec_ready=spec_ready, after_core=after_core, h32=h32)

    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 2
    ids = _ids(cfg, 1, 128, 30, gpu)
    model = _model(cfg, gpu, 31)
    want, _ = model(ids)
    for lay in model.encoder.layer:
        lay.__class__ = Plain
    for native in (True, False):
        model.encoder.native_schedule = native
        got, _ = model(ids)
        assert torch.equal(got, want)


def test_a_bad_index_is_reported_before_a_failing_pooler(gpu):
    """The flag of a forward with a bad id is read in that forward, whatever becomes of its pooler."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    model = _model(cfg, gpu, 32)
    ids = _ids(cfg, 1, 128, 33, gpu)
    want, _ = model(ids)
    bad = ids.clone()
    bad[0, 5] = cfg.vocab_size

    def fail(module, args):
        raise ArithmeticError("pooler")

    handle = model.pooler.register_forward_pre_hook(fail)
    with pytest.raises(IndexError):
        model(bad)
    with pytest.raises(ArithmeticError):
        model(ids)
    handle.remove()
    got, _ = model(ids)                                     # nothing is left of the bad id
    assert torch.equal(got, want)


def _captured(call):
    """(result tensors of a captured call, its graph); the call's Python side has run once, its kernels not at all."""
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        held = call()
    return held, graph


# the one-kernel MLP's and the streaming product's packed weights, first wanted by a capture after a forward of few rows
@pytest.mark.parametrize("helper,B", [("m2_bert_80m", 8), ("m2_bert_large", 3), ("m2_bert_large", 17)])
def test_copies_made_during_a_capture_are_not_kept(gpu, helper, B):
    import m2_amd
    cfg = getattr(m2_amd, helper)(128)
    cfg.num_hidden_layers = 2
    one, many = _ids(cfg, 1, 128, 34, gpu), _ids(cfg, B, 128, 35, gpu)
    want, _ = _model(cfg, gpu, 36)(many)
    model = _model(cfg, gpu, 36)
    model.encoder.native_schedule = False
    model.validate_ids = False
    first, _ = model(one)
    (held, _), graph = _captured(lambda: model(many))
    eager, _ = model(many)                                  # before any replay
    assert torch.equal(eager, want)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(held, want)
        assert torch.equal(model(one)[0], first)


def test_casts_made_during_a_capture_are_not_kept(gpu):
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    layer = m2_amd.BertLayer(cfg).to(gpu).eval()
    u = torch.randn(2, 128, 768, generator=torch.Generator().manual_seed(37)).to(gpu)
    u16 = u.bfloat16()
    with torch.no_grad():
        layer(u)                                            # the filters' table; no bf16 copy yet
        held, graph = _captured(lambda: layer(u16))
        eager = layer(u16)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(held, eager)
        other = m2_amd.BertLayer(cfg).to(gpu).eval()
        other.load_state_dict(layer.state_dict())
        assert torch.equal(other(u16), eager)


# after an eager forward of one sequence: a capture at another row count of the native schedule (with other MLP kernels), and one
# that the Python schedule serves; through the model and through the encoder
@pytest.mark.parametrize("helper,L,B", [("m2_bert_80m", 128, 2), ("m2_bert_80m", 128, 8), ("m2_bert_large", 128, 3), ("m2_bert_80m", 1024, 9),
                                        ("m2_bert_large", 128, 17)])
def test_capture_at_another_batch_size(gpu, helper, L, B):
    import m2_amd
    cfg = getattr(m2_amd, helper)(L)
    cfg.num_hidden_layers = 2
    one, many = _ids(cfg, 1, L, 38, gpu), _ids(cfg, B, L, 39, gpu)
    h = torch.randn(B, L, cfg.hidden_size, generator=torch.Generator().manual_seed(40)).to(gpu)
    ref = _model(cfg, gpu, 41)
    want, wenc = ref(many)[0], ref.encoder(h)[-1]
    model = _model(cfg, gpu, 41)
    model.validate_ids = False
    model.pooler = None
    first, _ = model(one)
    (held, _), graph = _captured(lambda: model(many))
    held_enc, graph_enc = _captured(lambda: model.encoder(h)[-1])
    assert torch.equal(model(many)[0], want)
    for _ in range(3):
        graph.replay()
        graph_enc.replay()
        torch.randn(512, 512, device=gpu) @ torch.randn(512, 512, device=gpu)
        torch.cuda.synchronize()
        assert torch.equal(held, want) and torch.equal(held_enc, wenc)
        assert torch.equal(model(one)[0], first)


def test_embeddings_replaced_as_a_module(gpu):
    """Another embeddings module in front of the same encoder, there and back, and two models that share an encoder."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    a, b = _model(cfg, gpu, 42), _model(cfg, gpu, 43)
    ids = _ids(cfg, 1, 128, 44, gpu)
    first, _ = a(ids)
    b.encoder = a.encoder
    other, _ = b(ids)
    assert torch.equal(a(ids)[0], first) and not torch.equal(other, first)
    mine, a.embeddings = a.embeddings, b.embeddings
    (got, _), (want, _) = _both(a, ids)
    assert torch.equal(got, want) and torch.equal(got, other)
    a.embeddings = mine
    assert torch.equal(a(ids)[0], first)


def test_a_dropped_plan_outlives_its_use_on_another_stream(gpu):
    """The memory of a plan that is dropped while another stream still reads it is not given out again before that stream is done."""
    import m2_amd
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 2
    model = _model(cfg, gpu, 45)
    model.validate_ids = False
    ids = _ids(cfg, 1, 128, 46, gpu)
    want = model(ids)[0].clone()
    a = torch.randn(8192, 8192, device=gpu, dtype=torch.bfloat16)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(200):
            b = a @ a
        got = model(ids)[0]
    plan = model.encoder._native_plans[128]
    address, like = plan.table.table.data_ptr(), plan.table.table.shape
    assert plan.routes[0][1].streams >= {side.cuda_stream} and plan.table._use.streams >= {side.cuda_stream}
    del plan
    model.encoder._native_plans.clear()
    new = [torch.full(like, 1, dtype=torch.int64, device=gpu) for _ in range(32)]
    assert not side.query(), "the other stream was done too early for this test to say anything"
    assert all(t.data_ptr() != address for t in new)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    del b


def test_plans_keep_no_replaced_weights(gpu):
    import m2_amd
    cfg = m2_amd.m2_bert_80m(256)
    cfg.num_hidden_layers = 1
    model = _model(cfg, gpu, 47)
    short, long = _ids(cfg, 1, 128, 48, gpu), _ids(cfg, 1, 256, 49, gpu)
    model(short), model(long)
    old = [weakref.ref(t) for p in model.encoder._native_plans.values() for t in p.keep]
    assert len(model.encoder._native_plans) == 2 and all(r() is not None for r in old)
    with torch.no_grad():
        for lin in (model.encoder.layer[0].attention.in_linear, model.encoder.layer[0].attention.out_linear,
                    model.encoder.layer[0].mlp.gated_layers, model.encoder.layer[0].mlp.wo):
            lin.weight.mul_(2)
    model(short)
    assert list(model.encoder._native_plans) == [128] and all(r() is None for r in old)
    model(long)
    assert len(model.encoder._native_plans) == 2
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 50))
    assert not model.encoder._native_plans
