"""One row in one launch (csrc/gemm_gemv.h) around the number of columns up to which a CU has one workgroup, whose columns' scalars are
requested in front of the quantize: the bits of the two-launch form."""
import numpy as np
import pytest
import torch

from test_gpu_one_launch_decode import _call, _layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# N, K, F, bits: two columns of every wave, more, one of some waves only, one column in all; int8 rows of 6400 bytes and longer
CASES = [(4096, 2048, 64, 4), (4104, 2048, 64, 4), (4089, 480, 0, 4), (2049, 1024, 32, 4), (2041, 1024, 32, 4), (9, 256, 32, 4), (1, 256, 32, 4),
         (4096, 6400, 32, 8), (4000, 6416, 48, 8), (4096, 15872, 256, 4)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("N,K,F,bits", CASES)
def test_same_bits_as_two_launches(N, K, F, bits, dtype):
    from quik_amd import _lib as L
    lib = L.load()
    rng = np.random.default_rng(N + K)
    mod, _, _, fi, _, _ = _layer(rng, N, K + F, F, bits, dtype, False)
    x = rng.standard_normal((1, K + F)).astype(np.float32)
    x[:, fi] *= 50
    xt = torch.from_numpy(x).to(DEV, dtype)
    out = []
    try:
        for mode in (1, 0):
            lib.quik_layer_set_one_launch(mode)
            out.append(_call(mod, xt, 0x5A))
    finally:
        lib.quik_layer_set_one_launch(1)
    assert bool((out[0][1] == 0x5A).all()) and not bool((out[1][1] == 0x5A).all())
    assert torch.equal(out[0][0].view(torch.int16), out[1][0].view(torch.int16))
