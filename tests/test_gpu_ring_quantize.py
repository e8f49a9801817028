"""fp16 rows of more than 16384 columns, more of them than CUs, into int8 operand buffers in tile order: the calls that go through
the LDS ring (quantize_tile8_ring_kernel in csrc/quantize.hip), at every number of groups per lane, without outlier columns and with as many
as lanes, at row lengths that are no multiple of a kilobyte, with workgroups of one to three rows, and the calls beside them that it
refuses.  Against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_long_row_quantize import _case, _check

pytestmark = pytest.mark.gpu


def _rows(beyond):
    return torch.cuda.get_device_properties(0).multi_processor_count + beyond


def _outliers(rng, n_in, F):
    """Adjacent ones, one whole group of 8, both ends of the row, the others anywhere."""
    if F < 32:
        return rng.permutation(n_in)[:F]
    fixed = np.array([0, 1, 2, 3, 4, 5, 6, 7, 8, 17, n_in - 1, n_in - 2, n_in - 9, 4096, 4097, 4103])
    return rng.permutation(np.concatenate([fixed, rng.permutation(np.setdiff1d(np.arange(n_in), fixed))[:F - len(fixed)]]))


# rows beyond the CUs, columns (columns / 8 / 512 rounded up: groups per lane), outlier columns
@pytest.mark.parametrize("beyond,n_in,F", [
    (1, 16384 + 64, 64),       # 5, most of the fifth past the row's end
    (9, 20480, 256),           # 5, exactly
    (9, 20480 - 64, 0),        # no outlier columns, no whole kilobytes
    (9, 20480 + 64, 64),       # 6
    (300, 24576, 128),         # 6, up to three rows per workgroup
    (9, 24576 + 64, 64),       # 7
    (70, 28672, 512),          # 7, as many outlier columns as lanes
    (9, 28672 + 96, 32),       # 8
    (9, 31744, 256),           # 8: the longest row whose ring fits the LDS
    (300, 31744, 256),
    (40, 30720 - 64, 0),
])
def test_rows_through_the_ring(beyond, n_in, F):
    rng = np.random.default_rng(beyond + n_in + F)
    x, ii, fi = _case(rng, _rows(beyond), n_in, _outliers(rng, n_in, F))
    _check(x, ii, fi, n_in)


@pytest.mark.parametrize("seed", range(8))
def test_random_shapes_through_the_ring(seed):
    rng = np.random.default_rng(2000 + seed)
    F = 32 * int(rng.integers(0, 17))
    n_in = 64 * int(rng.integers((16448 - F + 63) // 64, (31744 - F) // 64 + 1)) + F
    fi = rng.permutation(n_in)[:F] if seed % 2 else n_in - 1 - rng.permutation(2 * F)[:F]
    x, ii, fi = _case(rng, _rows(int(rng.integers(1, 200))), n_in, fi)
    _check(x, ii, fi, n_in)


# one outlier column in each of as many groups as lanes, of more than that; rows whose ring exceeds the LDS
@pytest.mark.parametrize("beyond,n_in,F", [(9, 28672, 512), (9, 28672, 1024), (9, 32768, 256)])
def test_the_last_calls_of_the_ring_and_the_first_beyond(beyond, n_in, F):
    rng = np.random.default_rng(n_in + F)
    x, ii, fi = _case(rng, _rows(beyond), n_in, np.arange(F) * 8 + rng.integers(0, 8, F))
    _check(x, ii, fi, n_in)


def test_signalling_nans_in_the_ring():
    """Skipped by minimum and maximum like quiet ones, also between a row's extremes."""
    rng = np.random.default_rng(8)
    rows, n_in = _rows(9), 28672
    x, ii, fi = _case(rng, rows, n_in, _outliers(rng, n_in, 256))
    xb = x.view(np.uint16)
    for r in range(9, rows):
        xb[r, ii[rng.integers(0, len(ii), 6)]] = [0x7C01, 0x7D00, 0xFC01, 0x7DFF, 0x7E00, 0xFDAB]
    for r in (10, rows - 1):                           # right behind the minimum, right in front of the maximum
        xb[r, ii[64:72]] = np.array([-900.0, 0, 0, 0, 0, 0, 0, 0], np.float16).view(np.uint16)
        xb[r, ii[65]] = 0x7C01
        xb[r, ii[128:136]] = np.array([0, 0, 0, 0, 0, 0, 0, 900.0], np.float16).view(np.uint16)
        xb[r, ii[134]] = 0xFD55
    _check(x, ii, fi, n_in)
