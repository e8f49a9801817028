"""The oracle skips a signalling NaN like a quiet one, whatever the number of rows."""
import numpy as np
import pytest

from oracle import quik_oracle as qo


@pytest.mark.parametrize("rows", [1, 9, 16, 33, 48, 265])
def test_signalling_nans_are_skipped(rows):
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, 2000)).astype(np.float16)
    for r in range(rows):
        x.view(np.uint16)[r, rng.integers(0, 2000, 6)] = [0x7C01, 0x7D00, 0xFC01, 0x7DFF, 0x7E00, 0xFDAB]
    quiet = np.where(np.isnan(x), np.float16(np.nan), x)
    ii, fi = np.arange(0, 2000, 2), np.arange(1, 2000, 2)
    for got, want in zip(qo.asym_quantize(x, ii, fi, 8)[:2], qo.asym_quantize(quiet, ii, fi, 8)[:2]):
        assert np.array_equal(got, want)
