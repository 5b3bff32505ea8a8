"""The one-kernel MLP on either side of the row count where its tiles change: a row's sums run in the same order in both."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [4096, 4097, 4104, 6150, 8191])
def test_rows_do_not_depend_on_the_tile(gpu, M):
    from m2_amd import ops
    d, I, nb = 768, 3072, 4
    g = torch.Generator(device=gpu).manual_seed(M)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu)      # noqa: E731
    x, bias = rn(M, d).bfloat16(), rn(d)
    wg, wo = (rn(nb, 2 * I // nb, d // nb) * 0.07).bfloat16(), (rn(nb, d // nb, I // nb) * 0.05).bfloat16()
    for dtype in (torch.bfloat16, torch.float32):
        whole = ops.mlp_fused(x, wg, wo, bias, x, out_dtype=dtype)
        few = torch.cat([ops.mlp_fused(p.contiguous(), wg, wo, bias, p.contiguous(), out_dtype=dtype) for p in x.split(1000)])
        assert torch.equal(whole, few)
