"""Register-streaming int4 layer GEMM (csrc/gemm_direct.h): every number of k-steps that a wave can have in front of, inside and
behind the whole rounds of its loop, with no, few, one round of and more outlier steps.  Same bits as the row-major kernels."""
import pytest
import torch

from test_gpu_register_streaming import _same_bits

pytestmark = pytest.mark.gpu
OUTLIERS = (0, 32, 64, 96, 192, 224, 256, 288, 544)
# 128-column groups: two steps each, dealt to four waves.  Rounds of 8 steps (64x32 tiles), of 4 (64x64 and 128x64)
LONG, SHORT = (1, 3, 15, 17, 18, 19, 20, 33, 34, 35, 36, 37), (1, 2, 3, 9, 10, 11, 12, 13, 17, 18, 19, 26)


@pytest.mark.parametrize("M,N,groups", [(50, 1000, k) for k in LONG] + [(60, 8200, k) for k in SHORT] + [(128, 8200, k) for k in SHORT])
def test_step_counts(M, N, groups):
    _same_bits(M, N, 128 * groups, OUTLIERS[groups % len(OUTLIERS)], 4, torch.bfloat16 if groups % 4 == 3 else torch.float16)
