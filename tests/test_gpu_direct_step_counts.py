"""Register-streaming int4 layer GEMM (csrc/gemm_direct.h): every number of k-steps that a wave can have in front of, inside and
behind the whole rounds of its loop, with no, few, one round of and more outlier steps, on each of the three tiles.  Same bits as
the row-major kernels, or as the 6-bit ones."""
import pytest
import torch

from test_gpu_four_bit_weights import _problem
from test_gpu_register_streaming import _same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
OUTLIERS = (0, 32, 64, 96, 192, 224, 256, 288, 544)
# 128-column groups: two steps each, dealt to four waves.  Rounds of 4 steps, 5 in registers
LONG, SHORT = (13, 15, 17, 18, 19, 20, 33, 34, 35, 36, 37), (1, 2, 3, 9, 10, 11, 12, 13, 17, 18, 19, 26)


def _tile(M, N, K, F):
    from quik_amd import _lib as L
    return L.load().quik_tile4_tile(M, N, K, F)


# (few integer steps are on 64x32 tiles where the outlier steps are many)
@pytest.mark.parametrize("groups,F", [(g, 512 + 32 * (g % 2)) for g in range(1, 13)] + [(g, OUTLIERS[g % 9]) for g in LONG])
def test_step_counts_64x32(groups, F):
    assert _tile(50, 1000, 128 * groups, F) == 64 << 16 | 32
    _same_bits(50, 1000, 128 * groups, F, 4, torch.bfloat16 if groups % 4 == 3 else torch.float16)


@pytest.mark.parametrize("groups", SHORT)
def test_step_counts_64x64(groups):
    F = OUTLIERS[groups % len(OUTLIERS)]
    assert _tile(60, 8200, 128 * groups, F) == 64 << 16 | 64
    _same_bits(60, 8200, 128 * groups, F, 4, torch.bfloat16 if groups % 4 == 3 else torch.float16)


@pytest.mark.parametrize("groups", [1, 2, 3, 4, 5, 6, 7, 8] + [g for g in SHORT if g > 8])
def test_step_counts_128x64(groups):
    """A shape of the ring kernels with its activation in 4 bits: the 128x64 tiles take it, whatever its length."""
    from quik_amd import asymmetric, matmul
    M, N, K, F = 1100, 8328, 128 * groups, OUTLIERS[groups % len(OUTLIERS)]
    dtype = torch.bfloat16 if groups % 4 == 3 else torch.float16
    assert _tile(M, N, K, F) == 0
    _, _, cm, x, qw, fw, g = _problem(M, N, K, F, groups, dtype)
    s_col = (torch.rand(N, 1, generator=g, device=DEV) * 0.009 + 0.001).to(dtype)
    w_red = torch.randn(1, N, generator=g, device=DEV).to(dtype)
    out = []
    for four in (True, False):
        xb, meta = asymmetric.quantize_mapped_fp6(x, cm, K, F, four)
        w = matmul.pack_weight_fp6(qw, fw, cm, four)
        out.append((matmul.mixed_linear_tile4 if four else matmul.mixed_linear_fp6)(xb, w, meta, s_col, w_red, None, M, N, K, F, dtype))
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
