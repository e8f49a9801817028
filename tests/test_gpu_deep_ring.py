"""Tile-ordered GEMMs with one tile per CU (rings of twelve or eight slots): 128x64 tiles on 6-bit weights, 128x128 and 256x128
ones on 4-bit (the layer), 6-bit (the stand-alone operations) and int8 weights; fewer steps than slots, exactly as many, one pair more, whole turns with every remainder, none and more
outlier steps than slots.  Same output bits as the row-major int8-MFMA kernels, which other tests hold against the oracle."""
import pytest
import torch

from test_gpu_register_streaming import six_bit_operands

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,F", [(128, 13824, 128, 0), (100, 13830, 640, 32), (128, 13824, 768, 288), (127, 13800, 896, 0),
                                     (120, 13824, 1536, 64), (128, 13001, 1792, 256), (300, 5120, 2688, 96), (257, 4544, 4416, 128)])
def test_same_bits_as_the_row_major_kernels(M, N, K, F, dtype):
    _same_bits(M, N, K, F, dtype, 4)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,F", [(200, 10240, 128, 0), (365, 8190, 640, 32), (250, 10201, 768, 288), (380, 8192, 896, 0),
                                     (300, 8192, 4736, 64), (520, 9100, 384, 32), (600, 9001, 1664, 128)])
def test_one_wide_tile_per_cu(M, N, K, F, bits):
    _same_bits(M, N, K, F, torch.float16, bits)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,F", [(1025, 8200, 256, 32), (1100, 8300, 640, 0), (1217, 8321, 768, 96), (1280, 8448, 128, 0),
                                     (257, 4545, 384, 64), (2049, 4097, 256, 0)])
def test_waves_past_the_last_row_and_column(M, N, K, F, bits):
    """1, 76, 193 or all rows and 1, 8, 108, 129 or all columns in the last tiles: whole waves without a result."""
    _same_bits(M, N, K, F, torch.bfloat16, bits)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,F", [(2000, 11003, 256, 32), (1500, 11002, 1792, 64), (777, 21012, 640, 0)])
def test_both_tile_widths_in_one_launch(M, N, K, F, bits):
    """256x256 tiles with six slots beside 256x128 ones with eight or twelve, which start behind the first columns of every
    vector; 208, 220 or 9 rows and 123, 122 or 20 columns in the last tiles."""
    _same_bits(M, N, K, F, torch.bfloat16 if M == 777 else torch.float16, bits)


def _same_bits(M, N, K, F, dtype, bits):
    from quik_amd.qlinear import MixedQLinear
    g = torch.Generator().manual_seed(M + N + K + F)
    fi = torch.randperm(K + F, generator=g)[:F]
    s_w = (torch.rand(N, 1, generator=g) * 0.009 + 0.001).to(dtype)
    W = (torch.randint(-8, 8, (N, K + F), generator=g).float() * (1 if bits == 4 else 15) * s_w.float()).to(dtype)
    lin = torch.nn.Linear(K + F, N, bias=True, dtype=dtype)
    mod = MixedQLinear.from_float(lin, W, s_w, None, fi, bits=bits).to(DEV)
    x = torch.randn(M, K + F, generator=g)
    x[:, fi] *= 50
    x = x.to(dtype).to(DEV)
    got = [mod(x) for _ in range(2)] + six_bit_operands(mod, x)
    assert mod._w6 is not None
    mod.six_bit_path = False
    want = mod(x)
    for o in got:
        assert torch.equal(o.view(torch.int16), want.view(torch.int16))
