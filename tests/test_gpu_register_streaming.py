"""The register-streaming layer GEMM (csrc/gemm_direct.h) at the edges of its tiles: fewer k-steps than waves, step counts
that leave the waves unequal shares, one row more or less than a 64-row block, ragged and odd column counts, tiles that
start in the second half of a weight block, none, few and more outlier steps than it keeps in flight, K split over
workgroups.  Int4 cases run on 4-bit weights (the layer) and on the 6-bit operands (their stand-alone operations).  Same output bits as the row-major int8-MFMA kernels, which other tests hold against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # M, N, K, F, bits
    (33, 8, 128, 0, 4), (64, 32, 128, 32, 4), (65, 33, 256, 64, 4), (63, 64, 384, 0, 4), (40, 95, 896, 288, 4),
    (64, 1024, 7936, 256, 4), (100, 96, 1152, 544, 4), (128, 200, 2048, 256, 4), (129, 4096, 640, 32, 4),
    (200, 1001, 1920, 96, 4), (64, 2056, 3840, 256, 4), (513, 136, 512, 64, 4),
    (33, 8, 64, 0, 8), (64, 32, 64, 32, 8), (65, 33, 192, 64, 8), (63, 64, 320, 0, 8), (40, 95, 832, 288, 8),
    (64, 1024, 5504, 256, 8), (100, 96, 1088, 544, 8), (129, 4096, 576, 32, 8), (200, 1001, 1856, 96, 8),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_same_bits_as_the_row_major_kernels(case, dtype):
    _same_bits(*case, dtype)


@pytest.mark.parametrize("case", [(64, 5120, 13568, 256, 8), (96, 20480, 7936, 256, 4), (40, 8192, 10752, 256, 8)])
def test_plans_of_large_weights(case):
    """66, 116 and 84 MB of weights: 64x64 tiles with two splits, the ring of 128x128 tiles, 64x32 tiles."""
    _same_bits(*case, torch.float16)


def six_bit_operands(mod, x):
    """The forward of an int4 layer on 6-bit weights and activations, where its shape has such buffers."""
    from quik_amd import asymmetric, matmul
    if mod.bits != 4 or mod.int_features_num % 128 != 0:
        return []
    K, F, cm = mod.int_features_num, mod.fp_features_num, mod._column_map()
    fp_w = mod.fp_weight if F else torch.empty(mod.out_features, 0, dtype=mod.dtype, device=DEV)
    x6, meta = asymmetric.quantize_mapped_fp6(x, cm, K, F)
    out = matmul.mixed_linear_fp6(x6, matmul.pack_weight_fp6(mod.int_weight, fp_w, cm), meta, mod.weights_scales, mod.reduced_w, mod.bias,
                                  x.shape[0], mod.out_features, K, F, mod.dtype)
    return [out[None]]


def _same_bits(M, N, K, F, bits, dtype):
    from quik_amd import matmul
    from quik_amd.qlinear import MixedQLinear
    g = torch.Generator().manual_seed(M + N + K + F + bits)
    fi = torch.randperm(K + F, generator=g)[:F]
    s_w = (torch.rand(N, 1, generator=g) * 0.009 + 0.001).to(dtype)
    lo, hi = (-8, 8) if bits == 4 else (-127, 128)
    W = (torch.randint(lo, hi, (N, K + F), generator=g).float() * s_w.float()).to(dtype)
    lin = torch.nn.Linear(K + F, N, bias=True, dtype=dtype)
    mod = MixedQLinear.from_float(lin, W, s_w, None, fi, bits=bits).to(DEV)
    x = torch.randn(M, K + F, generator=g)
    x[:, fi] *= 50
    x = x.to(dtype).to(DEV)
    got = [mod(x) for _ in range(2)]
    assert mod._w6 is not None
    got += six_bit_operands(mod, x)
    matmul.split_k = False
    try:
        got.append(mod(x))
        got += six_bit_operands(mod, x)
    finally:
        matmul.split_k = True
    mod.six_bit_path = False
    want = mod(x)
    for o in got:
        assert torch.equal(o.view(torch.int16), want.view(torch.int16))
