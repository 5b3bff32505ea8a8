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


def test_dense_unsupported_sizes_are_refused(gpu):
    from m2_amd import ops
    for M, N, K in ((12, 64, 64), (64, 20, 64), (64, 64, 96)):
        assert not ops.lib.m2_dense_supported(M, N, K)
        with pytest.raises(RuntimeError, match="multiples of 8"):
            ops.dense_to_channels(torch.zeros(M, K, dtype=torch.bfloat16, device=gpu),
                                  torch.zeros(N, K, dtype=torch.bfloat16, device=gpu))
