"""The two ways fp32 operands of the filter MLPs become 16-bit parts, restated on the CPU with the bounds that stand beside them
(m2_amd/csrc/hyena_filter.h): what the parts hold and what the products left out amount to."""
import numpy as np

RNG = np.random.default_rng(0)
# mantissas drawn evenly, and those that lie between two numbers of 8, 11 and 16 bits
X = np.concatenate([1 + RNG.random(400000), *(1 + (RNG.integers(0, 2 ** b, 50000) + 0.5 + RNG.normal(0, 1e-3, 50000)) * 2.0 ** -b
                                              for b in (7, 10, 15))]).astype(np.float32)
X = X[(X >= 1) & (X < 2)]


def _bf16(x):
    u = np.asarray(x, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)


def _three_bf16(x):
    hi = _bf16(x)
    mid = _bf16(x - hi)
    return [p.astype(np.float64) for p in (hi, mid, _bf16(x - hi - mid))]


def _two_fp16(x):
    hi = x.astype(np.float16)
    return [p.astype(np.float64) for p in (hi, (x - hi.astype(np.float32)).astype(np.float16))]


def test_three_bf16_parts_hold_every_fp32_value():
    for size in (2.0 ** -60, 1.0, 2.0 ** 60):
        x = X * np.float32(size)
        hi, mid, lo = _three_bf16(x)
        assert np.array_equal(hi + mid + lo, x.astype(np.float64))
        y = RNG.permutation(x)
        yh, ym, yl = _three_bf16(y)
        six = hi * yh + hi * ym + mid * yh + mid * ym + hi * yl + lo * yh
        exact = x.astype(np.float64) * y
        assert np.abs(six / exact - 1).max() <= 2.0 ** -24


def test_two_fp16_parts_and_three_products():
    x = X * np.float32(2.0 ** 12)
    hi, lo = _two_fp16(x)
    assert np.abs((hi + lo) / x.astype(np.float64) - 1).max() <= 2.0 ** -23
    y = RNG.permutation(x)
    yh, yl = _two_fp16(y)
    exact = x.astype(np.float64) * y
    assert np.abs(lo * yl / exact).max() <= 2.0 ** -22
    err = (hi * yh + hi * yl + lo * yh) / exact - 1
    assert np.abs(err).max() <= 2.0 ** -21
    even = slice(0, 400000)
    assert np.sqrt(np.mean(((_two_fp16(x[even])[0] + _two_fp16(x[even])[1]) / x[even].astype(np.float64) - 1) ** 2)) <= 2.0 ** -24
    # entries of a row smaller than its largest, which lies at 2^12: a low part is off by half of fp16's smallest step at most
    for octave in range(40):
        small = x * np.float32(2.0 ** -octave)
        hi, lo = _two_fp16(small)
        assert np.abs(hi + lo - small.astype(np.float64)).max() <= max(2.0 ** -23 * 2.0 ** (13 - octave), 2.0 ** -25)
