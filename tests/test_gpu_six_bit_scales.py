"""bf16 scales whose product s_row * s_col is finite in float32 while 64 times it is not: the tile-ordered kernels, which sum 64ths
of the integers, against the row-major ones, which sum the integers, bit for bit, and against the formula where the integer sum is 0."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows, columns: 64- and 128-row register-streaming tiles, 128x128 tiles one and two per CU, 256x128, 256x256 beside 256x128, 256x256
# alone, 256x256 with 128x128 behind whole rounds
@pytest.mark.parametrize("M,N", [(40, 1024), (300, 4544), (400, 5120), (1000, 4096), (600, 11000), (777, 22016), (2048, 8192),
                                 (2048, 10240)])
@pytest.mark.parametrize("F", [0, 64])
@pytest.mark.parametrize("every", [1, 97])     # every column, few of them among columns of ordinary scales
def test_scales_of_a_large_product(M, N, F, every):
    from quik_amd import asymmetric, matmul
    from quik_amd.qlinear import MixedQLinear
    K, dtype = 640, torch.bfloat16
    g = torch.Generator().manual_seed(M + N + F)
    fi = torch.randperm(K + F, generator=g)[:F]
    keep = torch.ones(K + F, dtype=torch.bool)
    keep[fi] = False
    ii = torch.arange(K + F)[keep]
    # columns by turns: no integer weight, one of +-1 or +-2
    W = torch.zeros(N, K + F)
    n = torch.arange(1, N, 2)
    W[n, ii[torch.randint(0, K, (len(n),), generator=g)]] = torch.tensor([-2.0, -1.0, 1.0, 2.0])[torch.randint(0, 4, (len(n),), generator=g)]
    W[:, fi] = 0.02 * torch.randn(N, F, generator=g)
    lin = torch.nn.Linear(K + F, N, bias=True, dtype=dtype)
    mod = MixedQLinear.from_float(lin, W.to(dtype), torch.ones(N, 1, dtype=dtype), None, fi, bits=4).to(DEV)
    x = torch.randn(M, K + F, generator=g) * 1e20
    x[:, fi] = torch.randn(M, F, generator=g)
    x = x.to(dtype).to(DEV)
    s_col = torch.rand(N, 1, generator=g) * 1e17 + 2e17
    few = torch.arange(N) % every != 0
    s_col[few] *= 1e-20
    mod.weights_scales.copy_(s_col.to(dtype))
    mod.reduced_w.zero_()
    got = mod(x)
    assert mod._w6 is not None
    cm = mod._column_map()
    q, meta, fp_x = asymmetric.quantize_mapped(x, cm, K, F, 4)
    product = meta.float().view(M, 2)[:, :1].double() * mod.weights_scales.double().view(1, N)[:, ::every]
    assert product.max() * 16 < 3.3e38 and product.min() * 64 > 3.5e38        # (codes of at most 8, weights of at most 2)
    fp_w = mod.fp_weight if F else torch.empty(N, 0, dtype=dtype, device=DEV)
    x6, meta6 = asymmetric.quantize_mapped_fp6(x, cm, K, F)
    six = matmul.mixed_linear_fp6(x6, matmul.pack_weight_fp6(mod.int_weight, fp_w, cm), meta6, mod.weights_scales, mod.reduced_w, mod.bias,
                                  M, N, K, F, dtype)
    matmul.split_k = False
    try:
        whole = mod(x)
    finally:
        matmul.split_k = True
    assert torch.isfinite(got).all()
    zero = (fp_x.double().view(M, F) @ fp_w.double().t() + mod.bias.double())[:, ::2]
    err = (got.view(M, N)[:, ::2].double() - zero).abs()
    assert (err <= 2.0 ** -8 * zero.abs() + 1e-6).all()          # one rounding to bf16, sums of 64 products in float32
    mod.six_bit_path = False
    want = mod(x).view(M, N).view(torch.int16)
    for out in (got, six, whole):
        assert torch.equal(out.reshape(M, N).view(torch.int16), want)
