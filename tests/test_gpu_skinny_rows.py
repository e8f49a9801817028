"""The weight-streaming kernel of at most 32 token rows (gemm_skinny.h) at the edges of its shares: the int32 product is exact, and
the fused form is the epilogue formula in float64 within the rounding of its fp32 steps and of the output."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FULL = 256                                   # compute units: shares of N / 256 columns, in steps of 4


def _codes(g, shape, bits):
    lo, hi = (-8, 8) if bits == 4 else (-128, 128)
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.int16).to(torch.int8)


def _packed(c, bits):
    if bits == 8:
        return c
    u = c.to(torch.int16) & 15
    return (u[:, 0::2] | u[:, 1::2] << 4).to(torch.uint8)


# token rows: blocks of 8 (copies) and 16 (products); columns: shares of 4, 16, 32, 48, 64, 96, 112 and a second round, ragged;
# K bytes: less than a chunk of 128, whole chunks, fewer and more than eight waves have, a tail of 16 to 112 bytes
SHAPES = [(1, 1, 32), (3, 7, 224), (8, 1030, 256), (9, 15 * FULL + 3, 4096), (16, 20 * FULL, 4096 + 32), (17, 33 * FULL + 1, 2304),
          (24, 48 * FULL, 2048 + 224), (25, 64 * FULL, 1792), (32, 64 * FULL + 4, 8192 - 32), (32, 4544, 12288 + 96),
          (16, 65 * FULL + 5, 4352), (5, 112 * FULL, 2048), (12, 112 * FULL + 4, 6400), (32, 100, 28672 - 256)]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int32_product_is_exact(M, N, K, bits):
    import quik
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a, b = _codes(g, (M, K), bits), _codes(g, (N, K), bits)
    want = (a.double() @ b.double().t()).to(torch.int32)
    mm = quik.matmul.int4Matmul if bits == 4 else quik.matmul.int8Matmul
    assert torch.equal(mm(_packed(a, bits), _packed(b, bits)), want)


# products of their own plan: more than 64 columns per CU and at most 8 rows in two rounds, whole and ragged; rows of 16 KB and more
# with three turns in flight (a wave's turns a multiple of three and one and two more, a tail)
@pytest.mark.parametrize("bits,M,N,kbytes", [(4, 8, 65 * FULL + 3, 1040), (8, 1, 80 * FULL - 9, 2048), (4, 9, 72 * FULL, 384), (8, 7, 112 * FULL, 128),
                                             (4, 3, 17 * FULL + 1, 16384), (8, 16, 4500, 16384 + 128 * 9), (4, 16, 5000, 18432 + 112),
                                             (8, 1, 32 * FULL - 2, 16384 + 16), (8, 17, 4500, 16384), (8, 4, 4400, 16384 - 16)])
def test_products_of_many_columns_and_of_long_rows(bits, M, N, kbytes):
    test_int32_product_is_exact(M, N, kbytes * 8 // bits, bits)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_fused_form(i, bits):
    from quik_amd import _lib
    M, N, K = SHAPES[i]
    M = max(M, 3)                            # (one and two rows are another kernel's)
    F = (0, 8, 24, 256, 264, 40, 520)[i % 7]
    bf16, symmetric, with_bias = i % 2 == 1, i % 3 == 2, i % 4 != 0
    dtype = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator(device=DEV).manual_seed(7 * M + N + K)
    a, b = _codes(g, (M, K), bits), _codes(g, (N, K), bits)
    fx, fw = (torch.randn(r, F, generator=g, device=DEV).to(dtype) for r in (M, N))
    sc, wr, bias = (torch.randn(N, generator=g, device=DEV).to(dtype) for _ in range(3))
    sc = sc * 2.0 ** -12
    meta = torch.rand(M, 1 if symmetric else 2, generator=g, device=DEV).add(0.1).to(dtype)
    out = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
    qa, qb = _packed(a, bits), _packed(b, bits)
    rc = _lib.load().quik_mixed_linear_fwd(
        _lib.ptr(qa), _lib.ptr(qb), _lib.ptr(meta), _lib.ptr(sc), None if symmetric else _lib.ptr(wr), _lib.ptr(fx) if F else None,
        _lib.ptr(fw) if F else None, _lib.ptr(bias) if with_bias else None, _lib.QUIK_BF16 if bf16 else _lib.QUIK_F16, M, N, K, F, bits,
        _lib.ptr(out), _lib.stream())
    assert rc == 0
    row = meta[:, :1].double()
    terms = [(a.double() @ b.double().t()) * row * sc.double()]
    outliers, magnitude = fx.double() @ fw.double().t(), fx.double().abs() @ fw.double().abs().t()
    if not symmetric:
        shift = 8 if bits == 4 else 128
        terms += [meta[:, 1:].double() * wr.double(), shift * row * wr.double()]
    if with_bias:
        terms += [bias.double().expand(M, N)]
    want = outliers + sum(terms)
    size = magnitude + sum(t.abs() for t in terms)
    # fp32: at most F additions of outlier products and eight more steps, each within 2^-24 of what has been added so far (times 2:
    # the product of the scales is rounded too); the output is rounded once, by at most
    # half a step of its 8 (bf16) or 11 (fp16) significant bits
    bound = 2 * (F + 8) * 2.0 ** -24 * size + (2.0 ** -8 if bf16 else 2.0 ** -11) * want.abs() + 2.0 ** -25
    assert bool(((out.double() - want).abs() <= bound).all())
