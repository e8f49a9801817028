"""Register-streaming int4 layer GEMM (csrc/gemm_direct.h): every number of k-steps that a wave can have in front of its loop's whole
rounds, on the tiles whose steps in flight depend on how many tiles there are: 64x64 tiles that share a CU, 128x64 tiles of at most two rows
of tiles.  The same bits as the 6-bit kernels."""
import pytest
import torch

from test_gpu_four_bit_weights import _problem

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _same_bits_as_six(M, N, K, F, dtype):
    from quik_amd import asymmetric, matmul
    _, _, cm, x, qw, fw, g = _problem(M, N, K, F, K, dtype)
    s_col = (torch.rand(N, 1, generator=g, device=DEV) * 0.009 + 0.001).to(dtype)
    w_red = torch.randn(1, N, generator=g, device=DEV).to(dtype)
    out = []
    for four in (True, False):
        xb, meta = asymmetric.quantize_mapped_fp6(x, cm, K, F, four)
        w = matmul.pack_weight_fp6(qw, fw, cm, four)
        out.append((matmul.mixed_linear_tile4 if four else matmul.mixed_linear_fp6)(xb, w, meta, s_col, w_red, None, M, N, K, F, dtype))
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


# 128-column groups: two steps each, dealt to four waves; rounds of two steps, three in registers
@pytest.mark.parametrize("M,N,F,groups", [(330, 3000, 288, 2), (130, 6000, 288, 3), (130, 8200, 288, 4), (130, 8200, 288, 5), (65, 8200, 288, 6),
                                          (330, 3000, 128, 7), (130, 6000, 128, 8), (65, 8200, 128, 9), (330, 3000, 32, 10), (257, 3500, 0, 11),
                                          (65, 8200, 0, 13), (34, 16500, 0, 19)])
def test_step_counts_64x64_sharing_a_cu(M, N, F, groups):
    from quik_amd import _lib as L
    assert L.load().quik_tile4_tile(M, N, 128 * groups, F) == 64 << 16 | 64 and (M + 63) // 64 * ((N + 63) // 64) > 256
    _same_bits_as_six(M, N, 128 * groups, F, torch.bfloat16 if groups % 4 == 3 else torch.float16)


# (the ring kernels' shapes with the activation in 4 bits: the widest tiles take them, whatever their length)
@pytest.mark.parametrize("groups", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 13])
def test_step_counts_128x64_of_few_rows(groups):
    from quik_amd import _lib as L
    M, N = (100, 16504) if groups % 2 else (250, 20008)
    F = (0, 32, 256, 288)[groups % 4]
    assert L.load().quik_tile4_tile(M, N, 128 * groups, F) == 0
    _same_bits_as_six(M, N, 128 * groups, F, torch.bfloat16 if groups % 4 == 3 else torch.float16)


# int8: steps of 32 columns, two per 64, dealt to four waves; rounds of six steps on 64x32 tiles, of four on 64x64 ones
@pytest.mark.parametrize("blocks", [1, 2, 3, 5, 8, 11, 12, 13, 14, 15, 17, 19, 21, 22, 24, 25, 26, 37])
def test_step_counts_int8(blocks):
    from test_gpu_register_streaming import _same_bits
    F, dtype = (0, 32, 256, 288)[blocks % 4], torch.bfloat16 if blocks % 3 == 2 else torch.float16
    _same_bits(50, 300, 64 * blocks, F, 8, dtype)
    _same_bits(60, 8200, 64 * blocks, F, 8, dtype)
