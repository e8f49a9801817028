"""Whole rounds of 256x256 tiles with a last round of 128x128 tiles in one launch: a rest of one column, of half a
tile, of as many tiles as CUs, ragged rows in both tile heights, a row count whose tiles do not divide the CUs.  Same output
bits as the row-major int8-MFMA kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,F,dtype", [(2048, 8192 + 8, 256, 32, torch.float16), (2048, 10240, 384, 0, torch.bfloat16),
                                           (1900, 8192 + 1025, 128, 64, torch.float16), (1025 + 256, 10752 + 264, 256, 0, torch.float16),
                                           (4096, 8192 + 600, 256, 32, torch.float16)])
def test_same_bits_as_the_row_major_kernels(M, N, K, F, dtype, bits):
    from quik_amd.qlinear import MixedQLinear
    g = torch.Generator().manual_seed(M + N + K + F)
    fi = torch.randperm(K + F, generator=g)[:F]
    s_w = (torch.rand(N, 1, generator=g) * 0.009 + 0.001).to(dtype)
    lo, hi = (-8, 8) if bits == 4 else (-127, 128)
    W = (torch.randint(lo, hi, (N, K + F), generator=g).float() * s_w.float()).to(dtype)
    lin = torch.nn.Linear(K + F, N, bias=True, dtype=dtype)
    mod = MixedQLinear.from_float(lin, W, s_w, None, fi, bits=bits).to(DEV)
    x = torch.randn(M, K + F, generator=g)
    x[:, fi] *= 50
    x = x.to(dtype).to(DEV)
    got = mod(x)
    assert mod._w6 is not None
    mod.six_bit_path = False
    assert torch.equal(got.view(torch.int16), mod(x).view(torch.int16))
