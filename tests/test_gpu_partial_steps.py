"""Layers whose integer columns do not fill whole k-steps of the tile-ordered path (4 bits: multiples of 32 that are no
multiple of 128, 8 bits: of 16 that are no multiple of 64): the operand buffers are filled up with zeros and the layer
takes the same kernels.  Same output bits as the row-major kernels; the unwritten positions of the activation buffer
hold whatever the workspace held (here: every pattern of a large fill)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # M, N, K, F, bits, symmetric: every remainder, every quantize kernel (a workgroup per row, streaming, LDS ring), GEMM tile and split
    (33, 40, 32, 0, 4, False), (64, 96, 160, 32, 4, False), (65, 1000, 4288, 256, 4, False), (300, 4544, 4416, 128, 4, False),
    (257, 520, 1248, 64, 4, True), (2048, 4096, 1056, 96, 4, False), (1500, 8200, 672, 32, 4, False),
    (64, 512, 8096, 96, 4, False), (1200, 300, 10848, 160, 4, False), (40, 96, 16480, 96, 4, False), (41, 64, 16416, 64, 4, True),
    (33, 40, 16, 0, 8, False), (64, 96, 80, 32, 8, False), (65, 1000, 4304, 256, 8, False), (300, 640, 11344, 256, 8, False),
    (2048, 4096, 1072, 96, 8, False), (100, 512, 20528, 480, 8, False),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_same_bits_as_the_row_major_kernels(case, dtype):
    from quik_amd.qlinear import MixedQLinear
    M, N, K, F, bits, symm = case
    if symm and dtype == torch.bfloat16:
        pytest.skip("symmetric activations are fp16")
    g = torch.Generator().manual_seed(sum(case))
    fi = torch.randperm(K + F, generator=g)[:F]
    s_w = (torch.rand(N, 1, generator=g) * 0.009 + 0.001).to(dtype)
    lo, hi = (-8, 8) if bits == 4 else (-127, 128)
    W = (torch.randint(lo, hi, (N, K + F), generator=g).float() * s_w.float()).to(dtype)
    lin = torch.nn.Linear(K + F, N, bias=True, dtype=dtype)
    mod = MixedQLinear.from_float(lin, W, s_w, None, fi, symm=symm, bits=bits).to(DEV)
    x = torch.randn(M, K + F, generator=g)
    x[:, fi] *= 50
    x = x.to(dtype).to(DEV)
    mod.six_bit_path = False
    want = mod(x)
    mod.six_bit_path = True
    filler = torch.arange(1 << 26, dtype=torch.int32, device=DEV).mul_(-1640531527)   # every byte pattern, freed below
    del filler
    got = mod(x)
    assert mod._w6 is not None
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert torch.equal(mod(x).view(torch.int16), want.view(torch.int16))
    lean = MixedQLinear.from_float(lin, W, s_w, None, fi, symm=symm, bits=bits).to(DEV)
    lean.transient_tiled_copy = True
    assert torch.equal(lean(x).view(torch.int16), want.view(torch.int16))
