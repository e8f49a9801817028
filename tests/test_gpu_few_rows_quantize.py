"""Quantize of a layer's few rows (quantize_few_rows_kernel in csrc/quantize.hip): codes, scales, zero points and outlier values of a
forward's workspace, bit for bit those of the stand-alone operation, which other tests hold against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_one_launch_decode import _call, _layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# rows, K, F, bits, outlier columns in runs: one, two, four and eight groups of eight columns per lane and their ends, more outlier columns than
# lanes, none, rows of less than a kilobyte; the last two are left to the other kernels (more gathered units than lanes, more rows)
CASES = [(2, 64, 32, 4, False), (3, 480, 32, 8, True), (16, 3840, 256, 4, False), (7, 4096, 8, 8, False), (32, 4064, 32, 4, True),
         (5, 8192, 8, 8, True), (4, 7936, 256, 4, False), (16, 13568, 256, 8, False), (3, 16128, 256, 4, False), (2, 16384, 8, 8, False),
         (3, 32512, 256, 8, False), (2, 32000, 768, 4, True), (9, 2048, 0, 8, False), (6, 4096, 1024, 4, False), (2, 31232, 1024, 4, False),
         (40, 2048, 64, 4, False)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,K,F,bits,runs", CASES)
def test_workspace_is_what_the_operation_gives(rows, K, F, bits, runs, dtype):
    from quik_amd import _lib as L, asymmetric
    lib = L.load()
    rng = np.random.default_rng(K + F + rows)
    mod, _, _, fi, ii, _ = _layer(rng, 16, K + F, F, bits, dtype, runs)
    x = rng.standard_normal((rows, K + F)).astype(np.float32)
    x[:, fi] *= 50
    x[0, ii[3]], x[0, ii[-1]] = np.nan, 9
    x[1, ii[K // 2]] = np.inf
    x[rows - 1] = 1.5
    if rows > 2:
        x[2, ii[0]], x[2, ii[-1]] = 6e4, -6e4
    xt = torch.from_numpy(x).to(DEV, dtype)
    lib.quik_layer_set_one_launch(0)
    try:
        _, ws = _call(mod, xt, 0x5A)
    finally:
        lib.quik_layer_set_one_launch(1)
    q, meta, fp_x = asymmetric.quantize_mapped(xt, mod._column_map(), K, F, bits)
    up = lambda n: (n + 255) // 256 * 256
    at = 0
    for want in (q, meta, fp_x):
        want = want.contiguous().view(torch.uint8).reshape(-1)
        assert torch.equal(ws[at:at + want.numel()], want)
        at += up(want.numel())
