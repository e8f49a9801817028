"""The column map's build at the edges of its passes: one mask word per thread up to 32768 columns (full and ragged last
words, one word, all of them), more columns than that, index lists in any order.  Codes, meta and outlier values of
the stand-alone quantize (which builds a map per call) and of the mapped one against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import quik_oracle as qo

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("order", ["ascending", "shuffled", "outliers first", "outliers last", "every eighth"])
@pytest.mark.parametrize("cols,num_fp", [(32, 2), (40, 8), (1064, 0), (1064, 40), (1050, 26), (8192, 256), (8224, 1024),
                                         (32768, 256), (32768, 32736), (32776, 64), (65560, 24)])
def test_index_lists_of_every_kind(cols, num_fp, order):
    import quik
    from quik_amd import asymmetric
    rng = np.random.default_rng(cols + num_fp)
    if order == "outliers first":
        fp = np.arange(num_fp)
    elif order == "outliers last":
        fp = np.arange(cols - num_fp, cols)
    elif order == "every eighth" and 8 * num_fp <= cols:
        fp = 8 * np.arange(num_fp)
    else:
        fp = rng.permutation(cols)[:num_fp]
    keep = np.ones(cols, bool)
    keep[fp] = False
    ii = np.arange(cols)[keep]
    if order == "shuffled":
        ii = rng.permutation(ii)
    x = rng.standard_normal((3, cols)).astype(np.float32)
    x[:, fp] *= 50
    x = x.astype(np.float16)
    xt, it, ft = (torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in (x, ii.astype(np.int64), fp.astype(np.int64)))
    want = qo.asym_quantize(x, ii, fp, 8)
    got = quik.asymmetric.quantize(xt, it, ft, 8)
    mapped = asymmetric.quantize_mapped(xt, asymmetric.build_colmap(it, ft, cols), len(ii), num_fp, 8)
    for a, b, w in zip(got, mapped, want):
        a, b = a.cpu().numpy(), b.cpu().numpy()
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
        assert np.array_equal(a.reshape(-1).view(np.uint8), np.ascontiguousarray(w).reshape(-1).view(np.uint8))
