"""Two token rows have two kernels, chosen by the number of columns (csrc/gemm_gemv.h, csrc/gemm_skinny.h).  A column comes out the
same on either: the members of a group, one call of all their columns, give the bits that each gives alone, and so do the one-launch
and the two-launch form of a layer."""
import pytest
import torch

from test_gpu_front_end import _module

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(autouse=True)
def _default_route():
    from quik_amd import _lib as L
    lib = L.load()
    lib.quik_layer_set_one_launch(-1)
    yield
    lib.quik_layer_set_one_launch(-1)


def _bits(t):
    return t.contiguous().view(torch.int16)


def _rows(n_in, fi, dtype, seed, special=None):
    x = torch.randn(2, n_in, generator=torch.Generator().manual_seed(seed))
    x[:, fi] *= 50
    if special is not None and len(fi):
        x[1, fi[-1]] = special
    return x.to(dtype).to(DEV)


# alone: the matrix-vector kernel for the narrow ones (at most 2048 columns), all of them, or none; together the other kernel
@pytest.mark.parametrize("sizes,n_in,F,bits", [((4096, 1024, 1024), 1024 + 256, 256, 4), ((1024, 1024, 1024), 2048 + 64, 64, 4),
                                               ((2048, 2048), 1600 + 512, 512, 8), ((10248, 10248), 512 + 288, 288, 4),
                                               ((800, 1500), 1536 + 32, 32, 8)])
def test_a_group_gives_the_bits_of_its_members(sizes, n_in, F, bits):
    from quik_amd.qlinear import SharedQuantizedInput
    shared = SharedQuantizedInput(len(sizes))
    mods = [_module(i, n, n_in, F, bits, shared) for i, n in enumerate(sizes)]
    alone = [_module(i, n, n_in, F, bits) for i, n in enumerate(sizes)]
    x = _rows(n_in, mods[0].fp_indices.cpu(), torch.float16, n_in)
    want = [a(x) for a in alone]
    for _ in range(2):
        for m, w in zip(mods, want):
            assert torch.equal(_bits(m(x)), _bits(w))


# outlier steps: none, a part of one, fewer than the eight partial sums, all of them, a second round begun and complete
@pytest.mark.parametrize("F", [0, 8, 40, 96, 256, 264, 384, 512])
@pytest.mark.parametrize("bits,dtype,special", [(4, torch.float16, None), (8, torch.bfloat16, None), (4, torch.bfloat16, float("inf")),
                                                (8, torch.float16, 65504.0)])
def test_one_launch_and_two(F, bits, dtype, special):
    from quik_amd import _lib as L
    lib = L.load()
    n_in = 672 + F
    mod = _module(F, 1200, n_in, F, bits)
    if dtype == torch.bfloat16:
        mod = mod.to(dtype)
    x = _rows(n_in, mod.fp_indices.cpu(), dtype, F, special)
    outs = []
    for mode in (1, 0, -1):
        lib.quik_layer_set_one_launch(mode)
        outs.append(mod(x))
    assert torch.equal(_bits(outs[0]), _bits(outs[1])) and torch.equal(_bits(outs[0]), _bits(outs[2]))
