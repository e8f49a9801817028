"""CPU check of the arithmetic of the bf16 quantize kernels: bf16(x / scale) by one multiplication with the fp32 reciprocal, and levels
without an upper clamp."""
import numpy as np


def _bf16(x):
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + (u >> 16 & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)


def test_one_product_rounds_like_the_quotient():
    """All pairs of 8-bit significands (a power of two changes nothing: no product on the fast path is subnormal before its level is 0),
    and exponents at the ends of the fast path."""
    d = (np.arange(128, 256, dtype=np.float32) / 128)[None, :]
    s = (np.arange(128, 256, dtype=np.float32) / 128)[:, None]
    for ed, es in ((0, 0), (3, 0), (-20, -19), (100, 97), (120, 120), (-60, -63)):
        dd, ss = d * np.float32(2.0) ** ed, s * np.float32(2.0) ** es
        got = _bf16(dd * (np.float32(1.0) / ss))
        exact = dd.astype(np.float64) / ss.astype(np.float64)
        m, e = np.frexp(exact)
        t = m * 256
        low, frac = np.floor(t), t - np.floor(t)
        assert np.abs(frac - 0.5).min() / 256 > 2.0 ** -18       # (never near a tie, so the comparison does not hang on one)
        assert np.array_equal(got.astype(np.float64), np.ldexp((low + (frac > 0.5)) / 256, e))


def test_four_bit_quotient_never_reaches_the_upper_clamp():
    """The largest range that rounds to each bf16 scale significand, its largest numerator, both roundings: below 15.5."""
    s = (np.arange(128, 257, dtype=np.float64) / 128)[:, None]
    r = 15 * s * (1 + np.linspace(-1, 1, 4001)[None, :] * 2.0 ** -8)             # ranges around 15 scale
    r = r.astype(np.float32)
    scale = _bf16(r / np.float32(15.0))
    d = _bf16(r)
    assert (_bf16(d * (np.float32(1.0) / scale)) < 15.5).all()
