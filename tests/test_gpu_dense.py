"""The dense projections between row-major and channel-major activations (m2_dense_*) against fp64 products of the same
bf16 operands, at the sizes where their tiles and their dispatch change."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bf16(g, *shape):
    return torch.randn(*shape, generator=g).bfloat16()


def _within_bf16(got, ref, absref):
    """One rounding to bf16 (half an ulp: 2^-9 of the value, taken twice for the rounding boundary) on an fp32
    accumulation whose error stays below 2^-20 of the sum of absolute products (K <= 2048 additions)."""
    err = (got.double().cpu() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + absref * 2.0 ** -20
    assert torch.isfinite(got).all()
    assert (err <= bound).all(), ((err - bound).max().item(), (err > bound).sum().item())


# (M, N, K): one row group, ragged rows and columns, each tile variant (few rows; 64-, 128-row tiles; 192-wide; the two
# 256-row ones), one and several rounds, an odd number of K steps, the smallest K
@pytest.mark.parametrize("M,N,K", [(8, 8, 64), (32, 48, 64), (128, 2304, 768), (136, 200, 192), (256, 2304, 768), (520, 2880, 960),
                                   (1024, 4608, 1536), (2056, 2304, 768), (4096, 2304, 768), (8192, 2304, 768),
                                   (2048, 5376, 1792), (16384, 768, 768), (7688, 1000, 960), (96, 256, 2112)])
def test_dense_projections(gpu, M, N, K):
    from m2_amd import ops
    assert ops.lib.m2_dense_supported(M, N, K)
    g = torch.Generator().manual_seed(M + N + K)
    x, w, bias = _bf16(g, M, K), _bf16(g, N, K), torch.randn(N, generator=g)
    ref = x.double() @ w.double().T
    absref = x.double().abs() @ w.double().abs().T
    _within_bf16(ops.dense_to_channels(x.to(gpu), w.to(gpu)).t(), ref, absref)
    xt = x.t().contiguous().to(gpu)
    _within_bf16(ops.dense_from_channels(xt, w.to(gpu)), ref, absref)
    _within_bf16(ops.dense_from_channels(xt, w.to(gpu), bias.to(gpu)), ref + bias.double(), absref + bias.double().abs())


# the product with its weights in registers: the fewest rows it takes, fewer and more slabs of 32 rows than row ranges, a last slab of
# 8, 16 and 24 rows, one group of channels and so many that an XCD holds no whole row range, one to three and many slabs per range
@pytest.mark.parametrize("M,N", [(512, 2304), (520, 2304), (904, 2304), (1800, 2304), (2712, 768), (5632, 2304), (3000, 256), (8200, 256),
                                 (1000, 9216), (31744, 2304), (16376, 2304)])
def test_dense_weights_in_registers(gpu, M, N):
    from m2_amd import ops
    g = torch.Generator(device=gpu).manual_seed(M + N)
    x, w = torch.randn(M, 768, generator=g, device=gpu).bfloat16(), torch.randn(N, 768, generator=g, device=gpu).bfloat16()
    n = torch.cat([torch.arange(min(N, 300)), torch.arange(N - 128, N)]).unique().to(gpu)      # every row of x against these channels
    got = ops.dense_to_channels(x, w)
    _within_bf16(got[n].t(), x.cpu().double() @ w[n].cpu().double().T, x.cpu().double().abs() @ w[n].cpu().double().abs().T)
    m = torch.cat([torch.arange(0, M, max(1, M // 70)), torch.arange(M - 40, M)]).unique().to(gpu)   # and every channel on these rows
    _within_bf16(got[:, m].t(), x[m].cpu().double() @ w.cpu().double().T, x[m].cpu().double().abs() @ w.cpu().double().abs().T)


def test_channels_with_a_gap_between_them(gpu):
    """The projection into rows further apart than their values, and the core reading such rows: bit for bit those of dense rows, on
    each of the core's kernels and both kernels of the projection."""
    from m2_amd import ops
    g = torch.Generator(device=gpu).manual_seed(3)
    assert ops.channels_row(32768, 768) == 32832 and ops.channels_row(16376, 768) == 16376 and ops.channels_row(8192, 960) == 8192
    for L, B, d in ((128, 2, 768), (2048, 4, 768), (4096, 1, 64), (8192, 1, 768), (16384, 2, 64), (32768, 1, 8)):
        M, row = B * L, B * L + 72
        x, w = (torch.randn(n, 768, generator=g, device=gpu).bfloat16() for n in (M, 3 * d))
        dense = ops.dense_to_channels(x, w)
        wide = ops.dense_to_channels(x, w, row)
        assert wide.shape == (3 * d, row) and torch.equal(wide[:, :M], dense)
        sw, sb, pb = (torch.randn(3 * d, *s, generator=g, device=gpu) for s in ((3,), (), ()))
        u = torch.randn(d, B, L, generator=g, device=gpu)
        spec = ops.filter_spectrum(*(torch.randn(d, 2 * L, generator=g, device=gpu) * 0.02 for _ in range(2)), None, None)
        gap = wide.clone()
        gap[:, M:] = float("nan")
        for dt in (torch.bfloat16, torch.float32):
            want = ops.mixer_core(dense.to(dt).view(3 * d, B, L), u, sw, sb, spec, B, L, d, proj_bias=pb)
            got = ops.mixer_core(gap.to(dt), u, sw, sb, spec, B, L, d, proj_bias=pb, row=row)
            assert torch.equal(got, want), (L, dt)
    with pytest.raises(RuntimeError, match="multiple of 8"):
        ops.dense_to_channels(x, w, 32769)


def test_dense_unsupported_sizes_are_refused(gpu):
    from m2_amd import ops
    for M, N, K in ((12, 64, 64), (64, 20, 64), (64, 64, 96)):
        assert not ops.lib.m2_dense_supported(M, N, K)
        with pytest.raises(RuntimeError, match="multiples of 8"):
            ops.dense_to_channels(torch.zeros(M, K, dtype=torch.bfloat16, device=gpu),
                                  torch.zeros(N, K, dtype=torch.bfloat16, device=gpu))


def _blockdiag(x, w):
    nb, q, p = w.shape
    return torch.cat([x[:, k * p:(k + 1) * p] @ w[k].T for k in range(nb)], dim=1)


# wo with bias and residual on the tile engine: few rows, 240-wide blocks, each tile variant, ragged rows
@pytest.mark.parametrize("M,nb,q,p", [(1, 4, 8, 64), (33, 4, 192, 768), (128, 4, 240, 960), (1000, 4, 384, 1536), (2049, 2, 448, 1792),
                                      (4100, 4, 384, 1536), (8192, 4, 384, 1536), (5000, 4, 448, 1792), (40, 2, 24, 2112)])
def test_blockdiag_linear_bf16(gpu, M, nb, q, p):
    from m2_amd import ops
    g = torch.Generator().manual_seed(M + p)
    x, w, res, bias = _bf16(g, M, nb * p), _bf16(g, nb, q, p) * 0.05, _bf16(g, M, nb * q), torch.randn(nb * q, generator=g)
    ref, absref = _blockdiag(x.double(), w.double()), _blockdiag(x.double().abs(), w.double().abs())
    _within_bf16(ops.blockdiag_linear(x.to(gpu), w.to(gpu)), ref, absref)
    _within_bf16(ops.blockdiag_linear(x.to(gpu), w.to(gpu), bias.to(gpu), res.to(gpu)), ref + bias.double() + res.double(),
                 absref + bias.double().abs() + res.double().abs())


def _glu(x, w):
    nb, q, p = w.shape
    h = _blockdiag(x.double(), w.double())
    gate, val = h[:, :nb * q // 2], h[:, nb * q // 2:]
    return torch.nn.functional.gelu(gate) * val, val


def _within_glu(got, ref, val):
    """The GELU polynomial's 2.5e-4 of the value and one bf16 rounding, as for the other GLU kernels."""
    err = (got.double().cpu() - ref).abs()
    assert (err <= ref.abs() * 2.0 ** -7 + 2.5e-4 * (val.abs() + 1)).all(), err.max()


# the gated product of few rows: block widths off 32, one row, the last row count of its range and one beyond it
@pytest.mark.parametrize("M,nb,q,p", [(1, 4, 96, 192), (128, 4, 1536, 192), (256, 4, 1920, 240), (257, 4, 1920, 240), (64, 4, 3072, 384),
                                      (137, 4, 3584, 448), (70, 2, 40, 504)])
def test_blockdiag_glu_few_rows(gpu, M, nb, q, p):
    from m2_amd import ops
    g = torch.Generator().manual_seed(M + p)
    x, w = _bf16(g, M, nb * p), _bf16(g, nb, q, p) * (3 / p ** 0.5)
    _within_glu(ops.blockdiag_glu(x.to(gpu), w.to(gpu)), *_glu(x, w))


# the streaming kernel with the chunks of a block row dealt to several workgroups: one tile, uneven runs (30 and 56 chunks
# over 5, 8 and 16), several rounds of a split
@pytest.mark.parametrize("M,d", [(300, 960), (1100, 960), (700, 1536), (2000, 1536), (10300, 1536), (500, 1792), (10240, 1792)])
def test_glu_stream_split_chunks(gpu, M, d):
    from m2_amd import ops
    g = torch.Generator().manual_seed(M + d)
    x, w = _bf16(g, M, d), _bf16(g, 4, 2 * d, d // 4) * (3 / (d / 4) ** 0.5)
    got = ops.glu_stream(x.to(gpu), w.to(gpu))
    tiled = ops.blockdiag_glu(x.to(gpu), w.to(gpu))
    rows = torch.cat([torch.arange(min(M, 40)), torch.arange(max(0, M - 140), M)]).unique()
    _within_glu(got[rows.to(gpu)], *_glu(x[rows], w))
    assert (got.float() - tiled.float()).abs().max() <= 2.0 ** -6 * tiled.float().abs().max()


def _unaligned(t):
    """The same values two bytes off a 16-byte address."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    off = next(k for k in range(8) if (buf.data_ptr() + k * t.element_size()) % 16 == t.element_size())
    return buf[off:off + t.numel()].view_as(t).copy_(t)


def test_unaligned_bf16_operands(gpu):
    """Weights that are views into a flat bf16 buffer, and inputs, residuals and outputs at any address: kernels that load 16 bytes at a
    time through LDS are not used for them, the results are those of aligned ones."""
    import m2_amd
    from m2_amd import ops
    g = torch.Generator().manual_seed(5)
    for M, nb, q, p in ((33, 4, 192, 768), (1000, 4, 384, 1536), (2049, 2, 448, 1792)):
        x, w, res, bias = _bf16(g, M, nb * p), _bf16(g, nb, q, p) * 0.05, _bf16(g, M, nb * q), torch.randn(nb * q, generator=g)
        ref, absref = _blockdiag(x.double(), w.double()), _blockdiag(x.double().abs(), w.double().abs())
        ref, absref = ref + bias.double() + res.double(), absref + bias.double().abs() + res.double().abs()
        xg, wg, rg, bg = x.to(gpu), w.to(gpu), res.to(gpu), bias.to(gpu)
        _within_bf16(ops.blockdiag_linear(_unaligned(xg), wg, bg, rg), ref, absref)
        _within_bf16(ops.blockdiag_linear(xg, _unaligned(wg), bg, rg), ref, absref)
        _within_bf16(ops.blockdiag_linear(xg, wg, bg, _unaligned(rg)), ref, absref)
        out = _unaligned(torch.empty(M, nb * q, dtype=torch.bfloat16, device=gpu))
        _within_bf16(ops.blockdiag_linear(xg, wg, bg, rg, out=out), ref, absref)
    layer = m2_amd.BertLayer(m2_amd.m2_bert_80m(128)).to(gpu).eval()
    u = torch.randn(2, 128, 768, generator=g).to(gpu).bfloat16()
    with torch.no_grad():
        want = layer(u).float()
        for lin in (layer.attention.in_linear, layer.attention.out_linear, layer.mlp.gated_layers, layer.mlp.wo):
            lin.weight = torch.nn.Parameter(_unaligned(lin.weight.detach().bfloat16()))
            assert lin.weight.data_ptr() % 16 == 2
        for got in (layer(u), layer(_unaligned(u))):
            assert (got.float() - want).norm() <= 1e-2 * want.norm()
