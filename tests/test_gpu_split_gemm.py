"""fp32 products by three bf16 parts (m2_split_*) against fp64, at the sizes where their tiles and their dispatch change, and no
further from it than fp32 products are."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(g, *shape):
    return torch.randn(*shape, generator=g)


def _blockdiag(x, w):
    nb, q, p = w.shape
    return torch.cat([x[:, k * p:(k + 1) * p] @ w[k].T for k in range(nb)], dim=1)


def _within(got, ref, absref, K):
    """Products left out are below 3 x 2^-25 of |x w| each; 6 K / 32 additions into the accumulator and 32-term sums inside the
    instruction, each good for 2^-23 of the sum of absolute products at worst: bounded by (K / 4 + 8) 2^-24 of it."""
    err = (got.double().cpu() - ref).abs()
    assert torch.isfinite(got).all()
    assert (err <= absref * (K / 4 + 8) * 2.0 ** -24).all(), (err / absref).max()
    assert err.norm() <= 1e-6 * ref.norm()


# one row group, ragged rows and columns, K off the chunks of 32, each tile, an odd number of chunks, one chunk
@pytest.mark.parametrize("M,N,K", [(4, 4, 4), (36, 20, 32), (132, 288, 96), (128, 2304, 768), (1000, 2880, 960), (2052, 2304, 768),
                                   (2560, 2304, 768), (1024, 5376, 1792), (4100, 768, 772)])
def test_split_projections(gpu, M, N, K):
    from m2_amd import ops
    g = torch.Generator().manual_seed(M + N + K)
    x, w, bias, res = _rand(g, M, K), _rand(g, N, K), _rand(g, N), _rand(g, M, N)
    ref, absref = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    xg = x.to(gpu)
    xs, xt = ops.split_rows(xg, channel_major=True)
    assert torch.equal(xt, xg.t()) and torch.equal(ops.split_channels(xt), xs)
    ws, _ = ops.split_rows(w.to(gpu))
    _within(ops.split_to_channels(xs, ws, M, N, K).t(), ref, absref, K)
    _within(ops.split_linear(xs, ws, M, 1, K, N), ref, absref, K)
    _within(ops.split_linear(xs, ws, M, 1, K, N, bias.to(gpu), res.to(gpu)), ref + bias.double() + res.double(),
            absref + bias.double().abs() + res.double().abs(), K)


# block-diagonal: one row, blocks off the chunks (240), each tile
@pytest.mark.parametrize("M,nb,q,p", [(1, 4, 64, 64), (33, 4, 192, 240), (257, 2, 128, 24), (2560, 4, 1536, 192), (700, 4, 3584, 448)])
def test_split_blockdiag_and_glu(gpu, M, nb, q, p):
    from m2_amd import ops
    g = torch.Generator().manual_seed(M + p)
    x, w, bias = _rand(g, M, nb * p), _rand(g, nb, q, p) / p ** 0.5, _rand(g, nb * q)
    h, habs = _blockdiag(x.double(), w.double()), _blockdiag(x.double().abs(), w.double().abs())
    xs, _ = ops.split_rows(x.to(gpu), nb)
    ws, _ = ops.split_rows(w.view(-1, p).to(gpu))
    _within(ops.split_linear(xs, ws, M, nb, p, q, bias.to(gpu)), h + bias.double(), habs + bias.double().abs(), p)
    I = nb * q // 2
    parts = ops.split_glu(xs, ws, M, nb, p, q).view(M, I // 32, 3, 32).float()
    got = (parts[:, :, 0] + parts[:, :, 1] + parts[:, :, 2]).view(M, I)
    ref = torch.nn.functional.gelu(h[:, :I]) * h[:, I:]
    # errors of either factor (|gelu'| < 1.13) and a few roundings of erf and the product
    e = (p / 4 + 8) * 2.0 ** -24
    bound = 1.2 * e * (habs[:, :I] * h[:, I:].abs() + habs[:, I:] * h[:, :I].abs()) + 2.0 ** -20 * (h[:, :I].abs() + 1) * h[:, I:].abs()
    assert ((got.double().cpu() - ref).abs() <= bound + 1e-12).all()


def test_split_is_no_further_off_than_fp32(gpu):
    from m2_amd import ops
    for M, K in ((512, 768), (512, 1792), (260, 192)):
        g = torch.Generator().manual_seed(K)
        x, w = _rand(g, M, K), _rand(g, 4, 256, K // 4)
        ref = _blockdiag(x.double(), w.double())
        own = ops.split_linear(ops.split_rows(x.to(gpu), 4)[0], ops.split_rows(w.view(-1, K // 4).to(gpu))[0], M, 4, K // 4, 256)
        old = ops.blockdiag_linear_f32(x.to(gpu), w.to(gpu))
        assert (own.double().cpu() - ref).norm() <= 1.02 * (old.double().cpu() - ref).norm()


def test_split_infinities_and_nan(gpu):
    """What is not finite, huge or below the parts' range comes out as fp32 arithmetic has it."""
    from m2_amd import ops
    g = torch.Generator().manual_seed(1)
    x, w = _rand(g, 128, 64), _rand(g, 64, 64).bfloat16().float()
    x[3, 5], x[7, 9], x[9, 1] = float("inf"), float("nan"), 3.4e38
    x[11, 0], x[11, 1] = float("inf"), -float("inf")
    w[2, 5], w[30, 4] = 0.0, -float("inf")
    w[:, 1] = w[:, 1].clamp(-0.9, 0.9)
    x[20] *= 1e-20
    ref = x.double() @ w.double().T
    for got in (ops.split_linear(ops.split_rows(x.to(gpu))[0], ops.split_rows(w.to(gpu))[0], 128, 1, 64, 64),
                ops.split_to_channels(ops.split_rows(x.to(gpu))[0], ops.split_rows(w.to(gpu))[0], 128, 64, 64).t()):
        got = got.double().cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        inf = torch.isinf(ref)
        assert torch.equal(got[inf], ref[inf]) and torch.equal(torch.isinf(got), inf)
        ok = torch.isfinite(ref)
        scale = (x.double().abs() @ w.double().abs().T)[ok]
        assert ((got[ok] - ref[ok]).abs() <= 1e-5 * scale).all()


def test_fp32_modules_follow_their_weights(gpu):
    """A changed weight is the one used; hooks and unaligned or non-contiguous inputs take their way."""
    import copy

    import m2_amd
    from oracle import m2_oracle as O
    cfg = m2_amd.m2_bert_80m(128)
    sd = m2_amd.seeded_state_dict(cfg, 3, what="mixer")
    mix = m2_amd.MonarchMixerSequenceMixing(768, l_max=128, bidirectional=True, hyena_emb_dim=5, hyena_filter_order=128,
                                            residual_long_conv=True, hyena_w=10)
    mix.load_state_dict(sd)
    mix = mix.to(gpu).eval()
    u = torch.randn(3, 128, 768, generator=torch.Generator().manual_seed(4))
    buf = torch.empty(u.numel() + 1, device=gpu)
    odd = buf[1:].view_as(u).copy_(u)                                          # 4 bytes off
    with torch.no_grad():
        for _ in range(2):
            want = O.mixer_forward(sd, "", u)
            a = mix(u.to(gpu))[0]
            assert ((a.cpu() - want).abs().max() / want.abs().max()) < 1e-4
            assert torch.equal(mix(odd)[0], a) and torch.equal(copy.deepcopy(mix)(u.to(gpu))[0], a)
            assert torch.equal(mix(u.to(gpu).transpose(0, 1).contiguous().transpose(0, 1))[0], a)
            sd["in_linear.weight"] = sd["in_linear.weight"] * 1.5
            sd["out_linear.weight"] = sd["out_linear.weight"] * 0.5
            mix.in_linear.weight.mul_(1.5)
            mix.out_linear.weight.mul_(0.5)
        with pytest.raises(RuntimeError), torch.enable_grad():
            mix(u.to(gpu).requires_grad_())
        mlp = m2_amd.BertLayer(cfg).to(gpu).eval().mlp
        x = torch.randn(5, 77, 768, generator=torch.Generator().manual_seed(5)).to(gpu)
        got = mlp(x)
        seen = []
        hook = mlp.wo.register_forward_hook(lambda m, i, o: seen.append(o.shape))
        hooked = mlp(x)
        hook.remove()
        assert seen and (got - hooked).abs().max() < 1e-5
        mlp.wo.weight.add_(0.01)
        assert (mlp(x) - got).abs().max() > 1e-4


# rows and chunks off the groups of 32 and 64, several blocks, one to three weights behind the activation
@pytest.mark.parametrize("M,nb,p,shapes", [(4, 1, 4, [(4, 4)]), (33, 4, 24, [(4, 40, 24), (2, 100)]), (2052, 1, 768, [(2304, 768), (768, 768), (1, 36)])])
def test_split_of_several_operands_at_once(gpu, M, nb, p, shapes):
    from m2_amd import ops
    g = torch.Generator().manual_seed(M)
    x, ws = _rand(g, M, nb * p).to(gpu), [_rand(g, *s).to(gpu) for s in shapes]
    one, _ = ops.split_rows(x, nb)
    parts, xt, *wparts = ops.split_rows(x, nb, channel_major=nb == 1, weights=ws)
    assert torch.equal(parts, one) and (xt is None or torch.equal(xt, x.t()))
    for w, got in zip(ws, wparts, strict=True):
        K = w.shape[-1]
        assert torch.equal(got, ops.split_rows(w.view(-1, K))[0])
        whole = got.view(-1, (K + 31) // 32, 3, 32).float().sum(2).view(w.numel() // K, -1)
        assert torch.equal(whole[:, :K], w.view(-1, K)) and not whole[:, K:].any()


@pytest.mark.parametrize("B", [2, 11])              # the mixer's projections by the library and by parts
def test_fp32_modules_read_the_weights_of_the_call(gpu, B):
    """Weights written through `.data`, computed anew per access, replaced at an old address, or changed between two replays of
    a captured graph: a result is always that of the weights as they are."""
    import copy

    import m2_amd
    from torch.nn.utils import parametrize
    cfg = m2_amd.m2_bert_80m(128)
    layer = m2_amd.BertLayer(cfg).to(gpu).eval()
    u = torch.randn(B, 128, 768, generator=torch.Generator().manual_seed(6)).to(gpu)
    linears = [layer.attention.in_linear, layer.attention.out_linear, layer.mlp.gated_layers, layer.mlp.wo]

    class Scaled(torch.nn.Module):
        factor = 1.0

        def forward(self, w):
            return w * self.factor

    def fresh():
        other = m2_amd.BertLayer(cfg).to(gpu).eval()
        other.load_state_dict({k: v.clone() for k, v in layer.state_dict().items()})
        return other(u)

    with torch.no_grad():
        got = layer(u)
        for lin in linears:
            lin.weight.data.mul_(1.25)
            before, got = got, layer(u)
            assert torch.equal(got, fresh()) and not torch.equal(got, before)
        for lin in linears:                                    # freed and made again: the address may come back
            for _ in range(2):
                old = lin.weight.detach()
                lin.weight = None
                values = (old * 0.9).cpu()
                del old
                lin.weight = torch.nn.Parameter(values.to(gpu))
            before, got = got, layer(u)
            assert torch.equal(got, fresh()) and not torch.equal(got, before)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            held = layer(u)
        for factor in (1.1, 0.8, 1.3):
            for lin in linears:
                lin.weight.mul_(factor)
            torch.randn(512, 512, device=gpu) @ torch.randn(512, 512, device=gpu)
            want = fresh()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(held, want), factor
        want = copy.deepcopy(layer)
        for m in (want.mlp.gated_layers, want.mlp.wo):          # a subclass, as parametrised modules are: the same way through the MLP
            m.__class__ = type("Other", (m2_amd.BlockdiagLinear,), {})
        for lin in linears:
            parametrize.register_parametrization(lin, "weight", Scaled())
        for factor in (1.0, 1.5, 0.5, 2.0, 0.75):
            for lin, other in zip(linears, (want.attention.in_linear, want.attention.out_linear, want.mlp.gated_layers, want.mlp.wo)):
                lin.parametrizations.weight[0].factor = factor
                other.weight.copy_(lin.parametrizations.weight.original * factor)
            assert torch.equal(layer(u), want(u)), factor


# either side of the rules that choose between parts and the fp32 kernels
@pytest.mark.parametrize("i,o,M", [(768, 6144, 677), (768, 6144, 679), (6144, 1536, 3), (3072, 768, 1357)])
def test_fp32_blockdiag_linear_by_size(gpu, i, o, M):
    import m2_amd
    from m2_amd import blockdiag
    lin = m2_amd.BlockdiagLinear(i, o, nblocks=4)
    nb, q, p = lin.weight.shape
    assert blockdiag._parts_pay(M, nb, q, p) == (M != 677)
    x = _rand(torch.Generator().manual_seed(M), M, i)
    w, b = lin.weight.detach().double(), lin.bias.detach().double()
    ref, absref = _blockdiag(x.double(), w) + b, _blockdiag(x.double().abs(), w.abs()) + b.abs()
    with torch.no_grad():
        got = lin.to(gpu)(x.to(gpu))
    # (the fp32 kernel: K / 4 additions of four products each)
    assert ((got.double().cpu() - ref).abs() <= absref * (p / 2 + 8) * 2.0 ** -24).all()


@pytest.mark.parametrize("L,B", [(128, 10), (128, 11)])
def test_fp32_mixer_by_size(gpu, L, B):
    import m2_amd
    from oracle import m2_oracle as O
    cfg = m2_amd.m2_bert_80m(L)
    sd = m2_amd.seeded_state_dict(cfg, 3, what="mixer")
    mix = m2_amd.MonarchMixerSequenceMixing(768, l_max=L, bidirectional=True, hyena_emb_dim=5, hyena_filter_order=128,
                                            residual_long_conv=True, hyena_w=10)
    mix.load_state_dict(sd)
    mix = mix.to(gpu).eval()
    assert (mix._fp32_parts(B * L) is not None) == (B == 11)
    u = torch.randn(B, L, 768, generator=torch.Generator().manual_seed(4))
    with torch.no_grad():
        want = O.mixer_forward(O.cast_state_dict(sd, torch.float64), "", u.double())
        got = mix(u.to(gpu))[0].double().cpu()
    assert (got - want).norm() <= 1.6e-5 * want.norm()          # fp32 sums, four times what is measured


def test_fp32_mlp_calls_what_stands_in_for_its_linears(gpu):
    """A dense layer, a module without a weight, a subclass and an instance with a forward of their own in the place of
    gated_layers or wo: called, as with any other nn.Module."""
    import m2_amd
    mlp = m2_amd.BertLayer(m2_amd.m2_bert_80m(128)).to(gpu).eval().mlp
    x = _rand(torch.Generator().manual_seed(9), 40, 768).to(gpu)

    class Doubled(m2_amd.BlockdiagLinear):
        def forward(self, v):
            return 2 * super().forward(v)

    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, v):
            return 2 * self.inner(v)

    with torch.no_grad():
        plain = mlp(x)
        w, b = mlp.wo.weight.clone(), mlp.wo.bias.clone()
        mlp.wo.weight.mul_(2)
        mlp.wo.bias.mul_(2)
        doubled = mlp(x)
        mlp.wo.weight.copy_(w)
        mlp.wo.bias.copy_(b)
        assert (plain - doubled).abs().max() > 1e-2
        inner = mlp.wo
        mlp.wo = Wrapped(inner)
        assert (mlp(x) - doubled).abs().max() < 1e-5
        mlp.wo = inner
        inner.__class__ = Doubled
        assert (mlp(x) - doubled).abs().max() < 1e-5
        inner.__class__ = m2_amd.BlockdiagLinear
        inner.forward = lambda v: 2 * m2_amd.BlockdiagLinear.forward(inner, v)
        assert (mlp(x) - doubled).abs().max() < 1e-5
        del inner.forward
        assert torch.equal(mlp(x), plain)
        dense = torch.nn.Linear(768, 6144, bias=False).to(gpu)
        for k in range(4):
            dense.weight.zero_() if k == 0 else None
            dense.weight[k * 1536:(k + 1) * 1536, k * 192:(k + 1) * 192] = mlp.gated_layers.weight[k]
        mlp.gated_layers = dense
        assert (mlp(x) - plain).abs().max() < 1e-4
