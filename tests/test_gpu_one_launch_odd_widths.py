"""One launch per decode call (csrc/gemm_gemv.h) at widths whose column-map tables end inside a 16-byte piece: the bits of the
two-launch form, and no workspace touched."""
import numpy as np
import pytest
import torch

from test_gpu_one_launch_decode import DEV, _call, _layer

pytestmark = pytest.mark.gpu

# rows, N, in, F, bits, dtype, outlier columns in runs: integer columns 32 .. 4000 beyond a multiple of 128, rows of 8 mod 32 columns
CASES = [
    (1, 64, 32, 0, 4, torch.float16, False), (2, 40, 16, 0, 8, torch.float16, False), (1, 1664, 1280, 64, 4, torch.float16, False),
    (2, 712, 3648, 256, 4, torch.float16, True), (1, 333, 4160, 256, 8, torch.bfloat16, False), (2, 208, 1000 + 24, 32, 4, torch.bfloat16, False),
    (1, 100, 480 + 8, 8, 4, torch.float16, False), (2, 72, 496 + 24, 24, 8, torch.float16, True), (1, 1000, 7232 + 40, 40, 8, torch.float16, False),
    (2, 1000, 12032 + 96, 96, 4, torch.float16, False),
]


@pytest.mark.parametrize("rows,N,n_in,F,bits,dtype,runs", CASES)
def test_same_bits_as_two_launches(rows, N, n_in, F, bits, dtype, runs):
    from quik_amd import _lib as L
    lib = L.load()
    rng = np.random.default_rng(rows + N + n_in + F + bits)
    mod, _, _, fi, _, _ = _layer(rng, N, n_in, F, bits, dtype, runs)
    x = rng.standard_normal((rows, n_in)).astype(np.float32)
    x[:, fi] *= 50
    x[rows - 1, n_in - 1] = 9
    xt = torch.from_numpy(x).to(DEV, dtype)
    lib.quik_layer_set_one_launch(1)
    out1, ws1 = _call(mod, xt, 0x5A)
    try:
        lib.quik_layer_set_one_launch(0)
        out2, ws2 = _call(mod, xt, 0x5A)
    finally:
        lib.quik_layer_set_one_launch(1)
    assert bool((ws1 == 0x5A).all()) and not bool((ws2 == 0x5A).all())
    assert torch.equal(out1.view(torch.int16), out2.view(torch.int16))


# (the last: long int4 rows, two launches on the matrix-vector kernel)
@pytest.mark.parametrize("N,K,one", [(4096, 512, True), (4104, 512, False), (20480, 512, False), (20488, 512, True), (4096, 1504, True),
                                     (2056, 1536, False), (2048, 1536, True), (2048, 6112, True), (2048, 6144, False), (100, 13120, False)])
def test_two_rows_take_one_launch_with_few_or_very_many_columns(N, K, one):
    from quik_amd import _lib as L
    from oracle import quik_oracle as qo
    lib = L.load()
    rng = np.random.default_rng(N)
    mod, W, s_w, fi, _, bias = _layer(rng, N, K + 32, 32, 4, torch.float16, False)
    x = rng.standard_normal((2, K + 32)).astype(np.float16)
    xt = torch.from_numpy(x).to(DEV)
    lib.quik_layer_set_one_launch(-1)
    try:
        out, ws = _call(mod, xt, 0x5A)
    finally:
        lib.quik_layer_set_one_launch(1)
    assert bool((ws == 0x5A).all()) == one
    want = qo.mixed_qlinear_forward(x, qo.from_float(W, s_w, fi, 4), 4, bias=bias)[0].astype(np.float64)
    assert np.abs(out.float().cpu().numpy() - want).max() <= 1e-2 * float(np.sqrt((want ** 2).mean()))  # as the one-launch tests
