"""LayerNorm kernels at the sizes where they can go wrong: row counts around the workgroups' 8 and 16 rows and around the
switch between one and two rows per wave (2048), widths of one piece, one LDS pass, a remainder pass and the limit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 7, 8, 9, 2041, 2048, 2049, 2063, 4097]


def reference(x, gamma, beta, eps):
    return torch.nn.functional.layer_norm(x.double(), (x.shape[1],), gamma.double(), beta.double(), eps)


@pytest.mark.parametrize("d", [64, 384, 448, 768, 960, 2048])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layernorm_row_counts_and_widths(dtype, d):
    from m2_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(11)
    gamma = torch.randn(d, generator=gen, device="cuda")
    beta = torch.randn(d, generator=gen, device="cuda")
    for M in ROWS:
        x = (torch.randn(M, d, generator=gen, device="cuda") * 3 + 1).to(dtype)
        o32, o16, ot = ops.layernorm(x, gamma, beta, 1e-12, True, True, True)
        ref = reference(x, gamma, beta, 1e-12)
        # fp32 statistics of at most 2048 values added in 6 + d / 64 steps: below 40 roundings of 6e-8
        assert ((o32.double() - ref).norm() / ref.norm()).item() < 2.5e-6, (M, d)
        assert torch.equal(ot.t(), o32) and torch.equal(o16, o32.bfloat16()), (M, d)
        for want in ((True, False, False), (False, True, True)):        # without the LDS pass / without the fp32 form
            got = ops.layernorm(x, gamma, beta, 1e-12, *want)
            assert all(torch.equal(a, b) for a, b in zip(got, (o32, o16, ot)) if a is not None), (M, d, want)


@pytest.mark.parametrize("B,L", [(1, 1), (1, 130), (16, 128), (17, 128), (3, 1024)])
def test_embed_layernorm_row_counts(B, L):
    from m2_amd import ops
    d = 768
    gen = torch.Generator(device="cuda").manual_seed(12)
    word, typ, pos = (torch.randn(n, d, generator=gen, device="cuda") for n in (500, 2, 1024))
    gamma, beta = torch.randn(d, generator=gen, device="cuda"), torch.randn(d, generator=gen, device="cuda")
    ids = torch.randint(0, 500, (B, L), generator=gen, device="cuda")
    tt = torch.randint(0, 2, (B, L), generator=gen, device="cuda")
    o32, o16, ot = ops.embed_layernorm(ids, tt, None, word, typ, pos, gamma, beta, 1e-12, True, True, True)
    rows = (word[ids] + typ[tt] + pos[:L][None]).view(B * L, d)
    ref = reference(rows, gamma, beta, 1e-12)
    assert ((o32.view(B * L, d).double() - ref).norm() / ref.norm()).item() < 2.5e-6
    assert torch.equal(ot.reshape(d, B * L).t(), o32.view(B * L, d)) and torch.equal(o16, o32.bfloat16())


@pytest.mark.parametrize("M,d", [(1, 64), (63, 128), (64, 64), (65, 192), (300, 768), (4097, 960)])
def test_input_forms(M, d):
    from m2_amd import ops
    base = torch.randn(M * d + 1, generator=torch.Generator(device="cuda").manual_seed(13), device="cuda")
    base[0], base[1], base[M * d - 1] = float("inf"), float("nan"), -0.0
    for x in (base[:-1].view(M, d), base[1:].view(M, d)):            # also rows that start off a 16-byte boundary
        h16, hT = ops.input_forms(x)
        ref = x.to(torch.bfloat16)
        assert torch.equal(h16.isnan(), ref.isnan()) and torch.equal(h16.nan_to_num(), ref.nan_to_num())
        assert torch.equal(hT.view(torch.int32), x.t().contiguous().view(torch.int32))
