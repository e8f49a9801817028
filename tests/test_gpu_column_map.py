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


def _lists(rng, cols, num_fp, order):
    """Outlier columns that lie close together (few dirty groups) or apart (many), integer columns ascending or not."""
    fp = np.arange(num_fp) if order == "close" else rng.permutation(cols)[:num_fp]
    keep = np.ones(cols, bool)
    keep[fp] = False
    ii = np.arange(cols)[keep]
    return (rng.permutation(ii) if order == "shuffled" else ii).astype(np.int64), fp.astype(np.int64)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("cols,num_fp", [(1064, 40), (8192, 256)])  # four waves per row, eight
@pytest.mark.parametrize("first,second", [("close", "apart"), ("apart", "close"), ("apart", "shuffled"), ("shuffled", "apart")])
def test_row_major_quantize_takes_the_map_that_is_there(cols, num_fp, first, second, bits):
    """A map at an address that the library knows becomes another one of the same shape: rebuilt between a capture and its
    replay, rebuilt by a replay, copied over.  The row-major quantize answers for the map that the device holds."""
    from quik_amd import _lib as L
    from quik_amd import asymmetric
    rng = np.random.default_rng(cols + bits)
    rows, num_int = 5, cols - num_fp
    x = (3 * rng.standard_normal((rows, cols))).astype(np.float16)
    xt = torch.from_numpy(x).to(DEV)
    lists = [_lists(rng, cols, num_fp, o) for o in (first, second)]
    index = [tuple(torch.from_numpy(a).to(DEV) for a in pair) for pair in lists]
    want = [[np.ascontiguousarray(w).reshape(-1).view(np.uint8) for w in qo.asym_quantize(x, *pair, bits)] for pair in lists]

    def check(got, which):
        torch.cuda.synchronize()
        for a, w in zip(got, want[which]):
            assert np.array_equal(a.cpu().numpy().reshape(-1).view(np.uint8), w)

    def build(cm, pair):
        L.check(L.load().quik_colmap_build(L.ptr(pair[0]), num_int, L.ptr(pair[1]), num_fp, cols, L.ptr(cm), L.stream()), "build")

    cm = asymmetric.build_colmap(*index[0], cols)
    asymmetric.colmap_streams(cm, num_int, num_fp)  # known from here on
    check(asymmetric.quantize_mapped(xt, cm, num_int, num_fp, bits), 0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = asymmetric.quantize_mapped(xt, cm, num_int, num_fp, bits)
    for which in (0, 1, 0, 1):  # rebuilt at its address, replayed
        build(cm, index[which])
        asymmetric.colmap_streams(cm, num_int, num_fp)
        graph.replay()
        check(held, which)
    given = tuple(t.clone() for t in index[0])
    builds = torch.cuda.CUDAGraph()
    with torch.cuda.graph(builds):
        build(cm, given)
    for which in (0, 1, 0):  # rebuilt by a replay, of which the host hears nothing
        for t, new in zip(given, index[which]):
            t.copy_(new)
        asymmetric.colmap_streams(cm, num_int, num_fp)
        builds.replay()
        check(asymmetric.quantize_mapped(xt, cm, num_int, num_fp, bits), which)
    maps = [asymmetric.build_colmap(*pair, cols) for pair in index]
    for which in (1, 0, 1):  # copied over
        cm.copy_(maps[which])
        check(asymmetric.quantize_mapped(xt, cm, num_int, num_fp, bits), which)
