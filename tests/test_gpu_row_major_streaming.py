"""The row-streaming integer GEMMs (csrc/gemm_rows.h) and the other routes of the stand-alone products above decode size,
at the edges of their tiles: half a stage, fewer stages than waves, unequal shares, one row or column more or less than a
tile, odd widths (no 16-byte stores), two rounds of tiles, 128-row tiles, the deep ring, wide and half-wide tiles in one
launch.  Integer sums equal a 64-bit product, the fused forms have the oracle's bits."""
import numpy as np
import pytest
import torch

from oracle import quik_oracle as qo

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [  # M, N, bytes of K per row, bits (0: both)
    (33, 1, 64, 0), (64, 8, 128, 0), (65, 63, 192, 0), (40, 65, 512, 0), (130, 136, 576, 0), (63, 4096, 640, 0),
    (256, 4001, 1088, 0), (97, 200, 2496, 0),
    (60, 64 * 260, 3072, 0), (255, 64 * 110 + 5, 3136, 4),     # 64x64 tiles, two rounds
    (100, 64 * 200, 3136, 8), (255, 64 * 101 + 3, 3072, 8),    # 128x64 tiles
    (300, 4500, 512, 0), (513, 2000, 832, 0),                  # ring kernels, 128x64 tiles
    (777, 5128, 256, 0), (1000, 8203, 2624, 0),                # large tiles, both widths
    # rows that end inside a stage, in every wave's share of it: nothing but the rest, one to five stages in front of it
    (33, 7, 16, 0), (64, 65, 112, 0), (70, 130, 144, 0), (40, 64, 32 * 9, 0), (129, 100, 416, 0), (100, 72, 5 * 128 + 80, 0),
    (130, 64 * 129, 1040, 0), (300, 64 * 61 + 3, 560, 0),      # the same on 128x64 tiles
    (200, 64 * 230, 240, 0), (600, 6700, 688, 0), (1100, 9000, 208, 0),  # and on several rounds, and on the plain kernels
    (1, 64, 64, 0), (1, 1001, 4096, 0), (32, 64 * 257, 176, 0), (17, 8, 1040, 0),  # decode sizes, the fused forms in one launch
    (130, 64 * 128, 1024, 4), (257, 64 * 85, 1088, 4), (130, 64 * 128, 3072, 8),  # 128x64 tiles, whole stages
]


def _operands(M, N, kbytes, bits, g):
    if bits == 8:
        a, b = (torch.randint(-128, 128, (n, kbytes), generator=g, device=DEV, dtype=torch.int16).to(torch.int8) for n in (M, N))
        return a, b, a, b
    a, b = (torch.randint(0, 256, (n, kbytes), generator=g, device=DEV, dtype=torch.int16).to(torch.uint8) for n in (M, N))

    def codes(t):
        t = t.to(torch.int16)
        lo, hi = t & 15, t >> 4
        both = torch.stack([lo, hi], -1).reshape(t.shape[0], -1)
        return torch.where(both > 7, both - 16, both)
    return a, b, codes(a), codes(b)


@pytest.mark.parametrize("M,N,kbytes,bits", [(m, n, k, b) for m, n, k, w in CASES for b in ((4, 8) if w == 0 else (w,))])
def test_products_and_fused_forms(M, N, kbytes, bits):
    import quik
    g = torch.Generator(device=DEV).manual_seed(M + N + kbytes)
    a, b, ca, cb = _operands(M, N, kbytes, bits, g)
    acc = (ca.double() @ cb.double().t().contiguous()).to(torch.int32)
    mm = quik.matmul.int4Matmul if bits == 4 else quik.matmul.int8Matmul
    assert torch.equal(mm(a, b), acc)

    def half(*shape):
        return (torch.rand(*shape, generator=g, device=DEV) * 0.1).half()
    s_row, s_col, zero, w_red, y = half(M, 1), half(1, N), -half(M, 1), half(1, N), half(M, N)
    host = [t.cpu().numpy() for t in (s_row, s_col, zero, w_red, y)]
    with np.errstate(all="ignore"):
        want = qo.asym_fused_dequantize(acc.cpu().numpy(), host[0], host[1], 8.0, host[2], host[3], host[4])
        want_sym = qo.sym_dequantize(acc.cpu().numpy(), host[0], host[1], host[4], 32)
    asym = quik.asymmetric.int4FusedDequantize if bits == 4 else quik.asymmetric.int8FusedDequantize
    sym = quik.symmetric.int4FusedDequantize if bits == 4 else quik.symmetric.int8FusedDequantize
    for got, w in ((asym(a, b, s_row, s_col, 8.0, zero, w_red, y), want), (sym(a, b, s_row, s_col, y), want_sym)):
        got = got.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(w))
        assert np.array_equal(got[~np.isnan(w)].view(np.uint16), w[~np.isnan(w)].view(np.uint16))


@pytest.mark.parametrize("M,N,kbytes", [(64, 128, 256), (63, 136, 144), (1, 512, 64), (257, 64 * 85, 1088), (130, 64 * 128, 1024)])
@pytest.mark.parametrize("off", [0, 1])
def test_fused_form_with_y_in_the_lds_or_not(M, N, kbytes, off):
    """Whole and partial column tiles of one call, y on a 16-byte boundary and two bytes behind one: the same bits as the
    product and the stand-alone dequantize."""
    import quik
    g = torch.Generator(device=DEV).manual_seed(M + N + off)
    a, b, _, _ = _operands(M, N, kbytes, 4, g)
    s_row, s_col = ((torch.rand(*s, generator=g, device=DEV) * 0.1).half() for s in ((M, 1), (1, N)))
    y = torch.randn(M * N + off, generator=g, device=DEV).half()[off:].view(M, N)
    got = quik.symmetric.int4FusedDequantize(a, b, s_row, s_col, y)
    want = quik.symmetric.dequantize(quik.matmul.int4Matmul(a, b), s_row, s_col, y.clone(), 32)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("bits,M,N,kbytes", [(4, 1, 512, 4080), (4, 16, 8192, 4096), (4, 17, 512, 4096), (4, 1, 8256, 4096),
                                             (4, 24, 4096, 5120), (4, 25, 4096, 5632), (4, 1, 4160, 5632), (8, 1, 320, 5104),
                                             (8, 8, 4096, 5120), (8, 9, 321, 8192), (8, 1, 4160, 8192), (8, 3, 1001, 11264),
                                             (4, 32, 4096, 11008), (4, 17, 8192, 4096), (4, 8, 4104, 5120), (8, 9, 4096, 7152),
                                             (8, 32, 600, 7168), (8, 9, 333, 5120)])
def test_few_rows_in_one_launch_or_two(bits, M, N, kbytes):
    """Both sides of the rule between the row-streaming tiles and product + epilogue: the same bits, with a workspace and
    without one (then the tiles take either), eager and replayed from a graph."""
    import quik
    from quik_amd import _lib as L
    g = torch.Generator(device=DEV).manual_seed(M + N + kbytes)
    a, b, ca, cb = _operands(M, N, kbytes, bits, g)
    K = kbytes * (2 if bits == 4 else 1)
    lib = L.load()
    two = kbytes >= (4096 if bits == 4 else 5120 if M <= 8 else 7168) if N <= 4096 else \
        bits == 4 and 4096 <= kbytes < 5120 and N <= 8192 and M <= 16
    assert lib.quik_fused_dequantize_acc_bytes(M, N, K, bits) == (M * N * 4 if two else 0)
    s_row, s_col, zero, w_red, y = ((torch.rand(*s, generator=g, device=DEV) * 0.1).half()
                                    for s in ((M, 1), (1, N), (M, 1), (1, N), (M, N)))
    acc = (ca.double() @ cb.double().t().contiguous()).to(torch.int32)
    host = [t.cpu().numpy() for t in (acc, s_row, s_col, zero, w_red, y)]
    with np.errstate(all="ignore"):
        want = qo.asym_fused_dequantize(host[0], host[1], host[2], 8.0, *host[3:])

    def check(out):
        got = out.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(got[~np.isnan(want)].view(np.uint16), want[~np.isnan(want)].view(np.uint16))
    op = quik.asymmetric.int4FusedDequantize if bits == 4 else quik.asymmetric.int8FusedDequantize

    def call():
        return op(a, b, s_row, s_col, 8.0, zero, w_red, y)
    check(call())
    out = torch.empty(M, N, dtype=torch.float16, device=DEV)
    L.check(lib.quik_asym_fused_dequantize(L.ptr(a), L.ptr(b), L.ptr(s_row), L.ptr(s_col), 8.0, L.ptr(zero), L.ptr(w_red), L.ptr(y),
                                           M, N, K, bits, None, L.ptr(out), L.stream()), "without a workspace")
    check(out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = call()
    for _ in range(3):
        held.zero_()
        call()
        graph.replay()
        check(held)
