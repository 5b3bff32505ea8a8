"""The mixer core and the plain long convolution against fp64 transforms, at row counts that leave row batches, workgroups and rounds
partly filled, and on either side of the rule that chooses a kernel at L = 8192."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _conv(a, k, D):
    k = k.double().clone()
    k[:, 0] += D.double()
    n = k.shape[-1]
    return torch.fft.irfft(torch.fft.rfft(a, n=n) * torch.fft.rfft(k, n=n)[:, None], n=n)[..., :a.shape[-1]]


@pytest.mark.parametrize("L,d,B", [(128, 8, 1), (128, 24, 7), (128, 768, 33), (256, 8, 9), (512, 16, 5), (1024, 8, 3), (2048, 8, 3), (4096, 8, 1),
                                   (8192, 8, 1), (8192, 256, 2), (8192, 256, 3), (16384, 8, 2), (32768, 8, 1)])
@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
def test_mixer_core_rows(gpu, L, d, B, act):
    from m2_amd import ops
    g = torch.Generator().manual_seed(L + d + B)
    taps = [torch.randn(d, 2 * L, generator=g) / L ** 0.5 for _ in range(2)]
    D = [torch.randn(d, generator=g) for _ in range(2)]
    xproj, u = torch.randn(3 * d, B, L, generator=g).to(act), torch.randn(d, B, L, generator=g)
    sw, sb, pb = (torch.randn(3 * d, *s, generator=g) for s in ((3,), (), ()))
    spec = ops.filter_spectrum(taps[0].to(gpu), taps[1].to(gpu), D[0].to(gpu), D[1].to(gpu))
    x = torch.nn.functional.pad(xproj.double() + pb.double()[:, None, None], (2, 0))
    s = sb.double()[:, None, None] + sum(sw.double()[:, k, None, None] * x[..., k:k + L] for k in range(3))
    first, second = _conv(s[:d] * s[2 * d:], taps[0], D[0]) * s[d:2 * d], _conv(u.double(), taps[1], D[1])
    # fp32: the roundings are independent, two and a half in a stage of each of the three transforms (signal, filter, back) and a
    # dozen in the convolutions, the gate and the factors; each is below 2^-25 of its value in the root mean square, and their
    # squares add up.  Twice that for what a few rows leave to chance.  bf16: the gate and the result are rounded to 2^-9, here
    # relative to a result of which they are a part
    stages = 3 * (L.bit_length() - 1)
    tol = 2 * (2.5 * stages + 12) ** 0.5 * 2.0 ** -25 if act == torch.float32 else 2.0 ** -8
    for second_signal in (True, False):
        y = ops.mixer_core(xproj.to(gpu), u.to(gpu) if second_signal else None, sw.to(gpu), sb.to(gpu), spec, B, L, d, proj_bias=pb.to(gpu))
        ref = first + second if second_signal else first
        assert (y.double().cpu() - ref).norm() <= tol * ref.norm()
    plain = ops.fftconv(u.to(act).to(gpu), spec, B, L, d).double().cpu()
    ref = _conv(u.to(act).double(), taps[0], D[0])
    assert (plain - ref).norm() <= tol * ref.norm()


def test_spectra_of_the_shortest_rows(gpu):
    """At L = 128 the filters' transform is rounded twice and not in every stage: what is left are the two transforms of the signal, 14
    stages of two and a half roundings of 2^-25 in the root mean square, and half a dozen others.  (With a filter transform in
    fp32 the 8192 rows come out at 2.1e-7.)"""
    from m2_amd import ops
    L, d, B = 128, 256, 32
    g = torch.Generator(device=gpu).manual_seed(0)
    k, x = torch.randn(d, 2 * L, generator=g, device=gpu), torch.randn(d, B, L, generator=g, device=gpu)
    y = ops.fftconv(x, ops.filter_spectrum(k, None, None, None), B, L, d)
    ref = _conv(x.double(), k, torch.zeros(d, device=gpu))
    assert (y - ref).norm() <= (2.5 * 14 + 6) ** 0.5 * 2.0 ** -25 * ref.norm()


@pytest.mark.parametrize("L,d,B", [(512, 768, 11), (2048, 768, 3), (4096, 768, 1), (8192, 768, 1)])
def test_rows_dealt_unevenly(gpu, L, d, B):
    """Row counts at which some workgroups take one batch of rows more than others: every row is there and is itself (the rows of fp64
    transforms; bound as above)."""
    from m2_amd import ops
    g = torch.Generator(device=gpu).manual_seed(L + B)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu)      # noqa: E731
    k, x = rn(d, 2 * L) / L ** 0.5, rn(d, B, L)
    y = ops.fftconv(x, ops.filter_spectrum(k, None, None, None), B, L, d)
    ref = _conv(x.double(), k, torch.zeros(d, device=gpu))
    tol = 2 * (2.5 * 3 * (L.bit_length() - 1) + 6) ** 0.5 * 2.0 ** -25
    assert ((y - ref).norm(dim=2) <= tol * ref.norm(dim=2)).all()


@pytest.mark.parametrize("L,d,B", [(1024, 8, 1), (1024, 24, 3), (2048, 16, 1), (4096, 768, 1), (4096, 8, 2), (8192, 16, 1), (8192, 768, 1), (16384, 8, 1)])
@pytest.mark.parametrize("nfilters", [1, 2])
def test_mixer_core_on_taps(gpu, L, d, B, nfilters):
    """The core that transforms its filters itself, in part filled workgroups and with workgroups that take several rows, against fp64 transforms
    and against the core on spectra, whose bits it has."""
    from m2_amd import ops
    g = torch.Generator(device=gpu).manual_seed(L + d + B)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu)      # noqa: E731
    taps, D = rn(nfilters, d, 2 * L) / L ** 0.5, rn(nfilters, d)
    row = B * L + 64
    xproj, u = rn(3 * d, row).bfloat16(), rn(d, B, L)
    sw, sb, pb = rn(3 * d, 3), rn(3 * d), rn(3 * d)

    class Table:
        fpm = nfilters

        def use_on(self, handle):
            pass

    for skips in (True, False):
        skip = torch.tensor([D[f].data_ptr() if skips else 0 for f in range(nfilters)], dtype=torch.int64).to(gpu)
        zero = torch.zeros_like(D)
        Ds = D if skips else zero
        x = torch.nn.functional.pad(xproj[:, :B * L].view(3 * d, B, L).double() + pb.double()[:, None, None], (2, 0))
        s = sb.double()[:, None, None] + sum(sw.double()[:, k, None, None] * x[..., k:k + L] for k in range(3))
        ref = _conv(s[:d] * s[2 * d:], taps[0], Ds[0]) * s[d:2 * d]
        if nfilters == 2:
            ref = ref + _conv(u.double(), taps[1], Ds[1])
        second = u if nfilters == 2 else None
        y = ops.mixer_core(xproj, second, sw, sb, ops.MixerTaps(taps, skip.data_ptr(), Table()), B, L, d, proj_bias=pb, row=row)
        spec = ops.filter_spectrum(taps[0], taps[1] if nfilters == 2 else None, Ds[0], Ds[1] if nfilters == 2 else None)
        z = ops.mixer_core(xproj, second, sw, sb, spec, B, L, d, proj_bias=pb, row=row)
        assert (y.double() - ref).norm() <= 2.0 ** -8 * ref.norm()      # (the gate and the result are rounded to 2^-9)
        assert torch.equal(y, z)


def test_core_on_taps_refuses(gpu):
    from m2_amd import ops
    L, d = 1024, 8
    x, taps = torch.randn(3 * d, 1, L, device=gpu), torch.randn(2, d, 2 * L, device=gpu)
    sw, sb = torch.randn(3 * d, 3, device=gpu), torch.randn(3 * d, device=gpu)

    class Table:
        fpm = 2

        def use_on(self, handle):
            pass

    filters = ops.MixerTaps(taps, None, Table())
    with pytest.raises(TypeError):
        ops.mixer_core(x, None, sw, sb, filters, 1, L, d)                       # fp32 rows read spectra
    with pytest.raises(ValueError):
        ops.mixer_core(x.bfloat16()[:, :, :512].contiguous(), None, sw, sb, filters, 1, 512, d)
    short = ops.MixerTaps(taps[:, :, :1024].contiguous(), None, Table())
    with pytest.raises(RuntimeError):
        ops.mixer_core(x.bfloat16()[:, :, :512].contiguous(), None, sw, sb, short, 1, 512, d)


@pytest.mark.parametrize("L", [1024, 2048, 4096, 8192, 16384])
def test_core_on_taps_beyond_ordinary_numbers(gpu, L):
    """The bits of the core on spectra also next to the ends of fp32 (products that only the factor 1 / L of a spectrum keeps below the upper one), and
    where a row has an infinity or a NaN."""
    from m2_amd import ops
    d, B = 64, 2
    g = torch.Generator(device=gpu).manual_seed(L)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu)      # noqa: E731
    taps, xproj, u = rn(2, d, 2 * L) / L ** 0.5, rn(3 * d, B, L).bfloat16(), rn(d, B, L)
    u[:16] *= 1e35
    u[16:32] *= 1e-37
    u[40, 0, 5], u[41, 1, 7] = float("inf"), float("nan")
    sw, sb = rn(3 * d, 3), rn(3 * d)

    class Table:
        fpm = 2

        def use_on(self, handle):
            pass

    y = ops.mixer_core(xproj, u, sw, sb, ops.MixerTaps(taps, None, Table()), B, L, d)
    z = ops.mixer_core(xproj, u, sw, sb, ops.filter_spectrum(taps[0], taps[1], None, None), B, L, d)
    assert torch.equal(torch.isnan(y), torch.isnan(z)) and torch.equal(y.nan_to_num(7.0), z.nan_to_num(7.0))
    assert bool(torch.isfinite(y[:40]).all()) and not bool(torch.isfinite(y[40, 0]).all())
