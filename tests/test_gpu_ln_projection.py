"""LayerNorm and in_linear of few rows as one kernel: the bits of the two kernels it stands for, at the edges of its tiles."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [768, 960, 1536, 1792])
@pytest.mark.parametrize("M", [8, 24, 32, 40, 128, 136, 256, 384])
def test_same_bits_as_two_kernels(gpu, M, d):
    from m2_amd import ops
    from m2_amd._lib import check, lib
    g = torch.Generator(device=gpu).manual_seed(M + d)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu)      # noqa: E731
    s, w = (rn(M, d) * 3 + 1).bfloat16(), (rn(3 * d, d) * 0.05).bfloat16()
    s[0] = 0.0                                                   # a row without variance
    gamma, beta, eps, row = rn(d), rn(d), 1e-12, M + 64
    for want_t in (True, False):
        out, hT = torch.full((3 * d, row), 7.0, device=gpu, dtype=torch.bfloat16), torch.full((d, M), 7.0, device=gpu)
        check(lib.m2_layernorm_to_channels_fwd(s.data_ptr(), gamma.data_ptr(), beta.data_ptr(), eps, w.data_ptr(), out.data_ptr(), row,
                                               hT.data_ptr() if want_t else None, M, 3 * d, d, ops._stream()))
        _, h16, want_hT = ops.layernorm(s, gamma, beta, eps, want_f32=False, want_bf16=True, want_channel_major=True)
        assert torch.equal(hT, want_hT) if want_t else bool((hT == 7.0).all())
        assert bool((out[:, M:] == 7.0).all())
        # the product alone, in fp64: one rounding to bf16 of sums in fp32
        ref = w.double() @ h16.double().t()
        bound = ref.abs() * 2.0 ** -8 + (w.double().abs() @ h16.double().abs().t()) * 2.0 ** -20
        assert ((out[:, :M].double() - ref).abs() <= bound).all()
        if lib.m2_layernorm_to_channels_supported(M, 3 * d, d):
            assert torch.equal(out[:, :M], ops.dense_to_channels(h16, w))      # the kernel that it replaces sums in the same order


def test_refused(gpu):
    from m2_amd import ops
    from m2_amd._lib import lib
    t = torch.zeros(4096, 768, device=gpu)
    call = lambda s, M, N, K, row: lib.m2_layernorm_to_channels_fwd(s, t.data_ptr(), t.data_ptr(), 1e-5, t.data_ptr(), t.data_ptr(), row, None, M, N, K, ops._stream())      # noqa: E731
    assert call(None, 128, 2304, 768, 128) and call(t.data_ptr(), 128, 768, 768, 128) and call(t.data_ptr(), 128, 2304, 768, 64)
    assert call(t.data_ptr(), 12, 2304, 768, 16) and call(t.data_ptr() + 2, 128, 2304, 768, 128) and call(t.data_ptr(), 128, 192, 64, 128)
    assert not lib.m2_layernorm_to_channels_supported(128, 192, 64) and not lib.m2_layernorm_to_channels_supported(4096, 2304, 768)
