"""Filter taps where the split weights and the tiles of their products can go wrong: rows of very different sizes, zero rows, widths
with fewer channel tiles than waves and with a remainder, lengths on either side of each kernel, against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _uneven(fn, d, g):
    """Weights of the implicit filters whose rows are of very different sizes."""
    with torch.no_grad():
        for name, p in fn.named_parameters():
            leaf = name.rsplit(".", 1)[-1]
            if "implicit_filter" not in name or leaf == "freq":
                continue
            p.normal_(0.0, 0.1, generator=g)
            if leaf == "weight" and p.shape[1] == 128:
                last = p.shape[0] == d
                # inner rows down to nothing, output rows over most of fp32's range, single large entries in both
                p.mul_(2.0 ** torch.randint(-50 if last else -20, 50 if last else 1, (p.shape[0], 1), generator=g))
                p[3] = 0.0
                p[5, 7] *= 64.0
                if not last:
                    p[9] *= 2.0 ** -60


def _reference(fn, L, dtype, bidirectional=True):
    from oracle import m2_oracle as O
    sd = {k: v.detach().cpu().to(dtype) for k, v in fn.state_dict().items()}
    fwd, rev = (O.hyena_filter_taps(sd, "", L, rev=r)[0].T if bidirectional or not r else None for r in (False, True))
    return O.bidirectional_kernel(fwd, torch.zeros_like(fwd) if rev is None else rev, L)


@pytest.mark.parametrize("L,d", [(128, 64), (1024, 64), (1088, 192), (1024, 320), (2048, 192)])
def test_taps_of_rows_of_any_size(gpu, L, d):
    import m2_amd
    g = torch.Generator().manual_seed(L + d)
    fn = m2_amd.HyenaFilter(d, emb_dim=5, order=128, seq_len=L, bidirectional=True, w=10)
    _uneven(fn, d, g)
    ref, ref32 = _reference(fn, L, torch.float64), _reference(fn, L, torch.float32).double()
    taps = fn.to(gpu).bidirectional_taps(L).double().cpu()
    assert torch.isfinite(taps).all()
    # channel by channel: products good to a few 2^-24 each, and what fp32 arithmetic itself makes of sin(10 x)
    norm = ref.norm(dim=1)
    err, err32 = (taps - ref).norm(dim=1), (ref32 - ref).norm(dim=1)
    assert (err <= 8 * 2.0 ** -24 * norm + 4 * err32).all(), (err / norm.clamp_min(1e-300)).max()
    assert not taps[3].any()


@pytest.mark.parametrize("bidirectional", [True, False])
@pytest.mark.parametrize("fpm", [1, 2])
@pytest.mark.parametrize("L", [128, 256, 512])
def test_spectra_of_rows_of_any_size(gpu, L, fpm, bidirectional):
    """The kernel that projects and transforms in one, on two mixers with such rows: against spectra of fp64 taps, channel by channel
    and filter by filter."""
    import m2_amd
    from m2_amd import ops
    d, g = 64, torch.Generator().manual_seed(L + fpm)
    fns = [m2_amd.HyenaFilter(d, emb_dim=5, order=128, seq_len=L, bidirectional=bidirectional, w=10) for _ in range(2 * fpm)]
    for fn in fns:
        _uneven(fn, d, g)
    refs = [[_reference(fn, L, t, bidirectional).float().to(gpu) for t in (torch.float64, torch.float32)] for fn in fns]
    groups = [fns[i:i + fpm] for i in range(0, 2 * fpm, fpm)]
    table = ops.FilterTable([[f.to(gpu).kernel_params("both") for f in m] for m in groups], [[None] * fpm] * 2, L, d, 128, 5)
    spectra = ops.mixer_filter_spectra(table, w_mod=1.0, shift=float(fns[0].modulation.shift)).view(2, d, 2, 2 * L).double()
    for m in range(2):
        for f in range(2):
            if f >= fpm:
                assert not spectra[m, :, f].any()
                continue
            want, want32 = (ops.filter_spectrum(t, None, None, None).view(d, 2, 2 * L)[:, 0].double() for t in refs[m * fpm + f])
            norm, err, err32 = want.norm(dim=1), (spectra[m, :, f] - want).norm(dim=1), (want32 - want).norm(dim=1)
            # as for the taps, and the roundings of either transform
            assert (err <= 12 * 2.0 ** -24 * norm + 4 * err32).all(), (m, f, (err / norm.clamp_min(1e-30)).max())
            assert not spectra[m, 3, f].any()


def test_taps_of_infinite_and_large_weights(gpu):
    """Finite weights of any size give finite taps, infinite ones poison their channel only."""
    import m2_amd
    L, d = 1024, 64
    fn = m2_amd.HyenaFilter(d, emb_dim=5, order=128, seq_len=L, bidirectional=True, w=10)
    with torch.no_grad():
        for w in (fn.implicit_filter[6].weight,):
            w[1] = 1e36
            w[2, 4] = float("inf")
            w[6, 8] = float("nan")
    taps = fn.to(gpu).bidirectional_taps(L).cpu()[:, :L]
    bad = ~torch.isfinite(taps).all(dim=1)
    assert bad[2] and bad[6] and int(bad.sum()) == 2


@pytest.mark.parametrize("L", [128, 1024])
def test_inner_layers_keep_all_bits(gpu, L):
    """Weights and activations of the inner layers whose mantissas lie between two numbers of 11 bits, one product per neuron and a last
    sine of arguments up to 128, which shows the relative error of that product: sine, two products and two more sines are five
    roundings of 2^-24 at most, below 2 x 2^-24 in the root mean square.  (Operands in two fp16 parts without the product of the low
    ones would be 2^-22 off, all in one direction.)"""
    import m2_amd
    d = n = 128
    g = torch.Generator().manual_seed(L)
    between = 1 + 0.97 * 2.0 ** -11
    sign = torch.randint(0, 2, (n,), generator=g) * 2.0 - 1
    b0 = (0.01 + 0.01 * torch.rand(n, generator=g)).float()
    w1 = (torch.asin(between * 2.0 ** -7 * sign.double()) / torch.sin(b0.double())).float()
    w2 = between * 2.0 ** torch.randint(12, 15, (n,), generator=g).float()
    fn = m2_amd.HyenaFilter(d, emb_dim=5, order=n, seq_len=L, bidirectional=True, w=1)
    with torch.no_grad():
        for name, p in fn.named_parameters():
            if "implicit_filter" in name and not name.endswith("freq"):
                p.zero_()
        fn.modulation.deltas.zero_()
        for mlp in (fn.implicit_filter, fn.implicit_filter_rev):
            mlp[0].bias.copy_(b0)
            mlp[2].weight.copy_(torch.diag(w1))
            mlp[4].weight.copy_(torch.diag(w2))
            mlp[6].weight.copy_(torch.eye(n))
    taps = fn.to(gpu).bidirectional_taps(L).double().cpu()
    arg = w2.double() * torch.sin(w1.double() * torch.sin(b0.double()))
    err = (taps - torch.sin(arg)[:, None]) / arg[:, None]
    assert err.pow(2).mean().sqrt() <= 2 * 2.0 ** -24


@pytest.mark.parametrize("L", [128, 1024])
def test_inner_layers_round_their_sums_once_a_step(gpu, L):
    """Sums of 128 positive products whose last sine, at arguments around 90, shows the sums' relative error.  The leading products
    of a sum are added in eight steps, each a rounding (0.41 x 2^-24 in the root mean square) of what is there by then:
    0.82 sqrt(sum (k / 8)^2) = 1.3 x 2^-25; the other 40 products are added apart.  (In one sum, 48 roundings would leave 3 x 2^-25.)"""
    import m2_amd
    d = n = 128
    g = torch.Generator().manual_seed(L)
    b0 = 0.01 + 0.01 * torch.rand(n, generator=g)
    w1, w2 = 0.9 + 0.2 * torch.rand(n, generator=g), 32.0 + 32.0 * torch.rand(n, n, generator=g)
    fn = m2_amd.HyenaFilter(d, emb_dim=5, order=n, seq_len=L, bidirectional=True, w=1)
    with torch.no_grad():
        for name, p in fn.named_parameters():
            if "implicit_filter" in name and not name.endswith("freq"):
                p.zero_()
        fn.modulation.deltas.zero_()
        for mlp in (fn.implicit_filter, fn.implicit_filter_rev):
            mlp[0].bias.copy_(b0)
            mlp[2].weight.copy_(torch.diag(w1))
            mlp[4].weight.copy_(w2)
            mlp[6].weight.copy_(torch.eye(n))
    taps = fn.to(gpu).bidirectional_taps(L).double().cpu()
    arg = w2.double() @ torch.sin(w1.double() * torch.sin(b0.double()))
    err = (taps - torch.sin(arg)[:, None]) / arg[:, None]
    assert err.pow(2).mean().sqrt() <= 1.5 * 2.0 ** -25


@pytest.mark.parametrize("L,d", [(128, 64), (1024, 64)])
def test_arguments_without_a_sine_left(gpu, L, d):
    """fp32 arguments beyond 3e7 leave the sines wrong, but the taps finite and no larger than sines make them, on every route; NaN
    stays NaN."""
    import m2_amd
    g = torch.Generator().manual_seed(L)
    mixer = m2_amd.MonarchMixerSequenceMixing(d, l_max=L, bidirectional=True, hyena_emb_dim=5, hyena_filter_order=128,
                                              residual_long_conv=True)
    fn = mixer.filter_fn
    with torch.no_grad():
        for f in (fn, mixer.filter_fn2):
            for mlp in (f.implicit_filter, f.implicit_filter_rev):
                mlp[4].weight.normal_(0.0, 1.0, generator=g).mul_(10.0 ** torch.randint(6, 12, (128, 1), generator=g))
    most = torch.stack([m[6].weight.detach().abs().sum(1) for m in (fn.implicit_filter, fn.implicit_filter_rev)]).amax(0).to(gpu)
    mixer = mixer.to(gpu)
    taps = fn.bidirectional_taps(L)
    assert (taps.abs() <= 1.001 * most[:, None] * (1 + abs(float(fn.modulation.shift)))).all()
    assert torch.isfinite(mixer.filter_spectrum(L)).all()
    with torch.no_grad():
        fn.implicit_filter[4].bias[0] = float("nan")
    assert not torch.isfinite(fn.bidirectional_taps(L)[:, :L]).any()


@pytest.mark.parametrize("bidirectional", [True, False])
@pytest.mark.parametrize("fpm", [1, 2])
@pytest.mark.parametrize("L", [128, 256, 512])
def test_spectra_of_many_mixers_at_once(gpu, L, fpm, bidirectional):
    """Enough mixers for workgroups of 32 channels: the same bits as one mixer at a time, whose workgroups have 16."""
    import m2_amd
    from m2_amd import ops
    d, n = 768, 6
    torch.manual_seed(L + fpm)
    mixers = [m2_amd.MonarchMixerSequenceMixing(d, l_max=L, bidirectional=bidirectional, hyena_emb_dim=5, hyena_filter_order=128,
                                                residual_long_conv=fpm == 2).to(gpu) for _ in range(n)]
    entries = [m.filter_table_entry() for m in mixers]
    table = ops.FilterTable([e[0] for e in entries], [e[1] for e in entries], L, d, 128, 5)
    together = ops.mixer_filter_spectra(table)
    for i in range(n):
        assert torch.equal(together[i], ops.mixer_filter_spectra(table, first=i, count=1)[0])
