"""A NaN in a bf16 result is 0x7FC0 whatever its sign and payload were, on every kernel that a call can take: the bits of a
result do not depend on the number of rows or on the operands' order."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NANS = [0x7FC0, 0x7FFF, 0x7F81, 0xFFC0, 0xFFC1, 0xFF81, 0xFFFF]  # quiet and signalling, both signs


def _bf16(bits):
    return torch.tensor([b - 0x10000 if b & 0x8000 else b for b in bits], dtype=torch.int16).view(torch.bfloat16)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M", [1, 2, 16, 40, 128, 300, 1100])
def test_nans_of_a_bias(M, bits):
    from quik_amd.qlinear import MixedQLinear
    N, K, F = 1100, 1024, 64
    g = torch.Generator().manual_seed(M + bits)
    fi = torch.randperm(K + F, generator=g)[:F]
    s_w = (torch.rand(N, 1, generator=g) * 0.009 + 0.001).bfloat16()
    W = (torch.randint(-8, 8, (N, K + F), generator=g).float() * s_w.float()).bfloat16()
    lin = torch.nn.Linear(K + F, N, bias=True, dtype=torch.bfloat16)
    at = torch.randperm(N, generator=g)[:len(NANS)]
    with torch.no_grad():
        lin.bias[at] = _bf16(NANS)
    mod = MixedQLinear.from_float(lin, W, s_w, None, fi, bits=bits).to(DEV)
    x = torch.randn(M, K + F, generator=g).bfloat16().to(DEV)
    for six_bit_path in (True, False):
        mod.six_bit_path = six_bit_path
        out = mod(x).reshape(M, N).cpu()
        assert torch.equal(out.view(torch.int16)[:, at], torch.full((M, len(NANS)), 0x7FC0, dtype=torch.int16))
        assert int(out.isnan().sum()) == M * len(NANS)


@pytest.mark.parametrize("bits", [4, 8])
def test_nans_of_a_dequantized_sum(bits):
    from quik_amd import asymmetric
    rows, cols = 9, 72
    g = torch.Generator().manual_seed(bits)
    acc = torch.randint(-1000, 1000, (rows, cols), generator=g, dtype=torch.int32)
    meta = torch.rand(2 * rows, generator=g).bfloat16()
    sc, wr = torch.rand(cols, 1, generator=g).bfloat16(), torch.rand(1, cols, generator=g).bfloat16()
    y = torch.randn(rows, cols, generator=g).bfloat16()
    y[:, :len(NANS)] = _bf16(NANS)
    out = asymmetric.dequantize(*(t.to(DEV) for t in (acc, meta, sc, wr, y)), bits).cpu()
    assert torch.equal(out.view(torch.int16)[:, :len(NANS)], torch.full((rows, len(NANS)), 0x7FC0, dtype=torch.int16))
    assert int(out.isnan().sum()) == rows * len(NANS)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,F", [(1280, 13056, 0), (2000, 11003, 32), (2048, 10240, 0), (300, 9000, 0), (520, 4100, 32)])
def test_nans_of_every_operand_on_large_tiles(M, N, F, bits):
    """Tiles of 256x256, of both widths in one launch, with 128x128 ones behind whole rounds, one 128x128 or 128x64 tile per CU:
    NaNs of the scales, the reduced weights, the bias and a row's outlier values, everything else the same bits as the
    row-major kernels."""
    from quik_amd.qlinear import MixedQLinear
    K = 128
    g = torch.Generator().manual_seed(M + bits)
    fi = torch.randperm(K + F, generator=g)[:F]
    s_w = (torch.rand(N, 1, generator=g) * 0.009 + 0.001).bfloat16()
    W = (torch.randint(-8, 8, (N, K + F), generator=g).float() * s_w.float()).bfloat16()
    lin = torch.nn.Linear(K + F, N, bias=True, dtype=torch.bfloat16)
    mod = MixedQLinear.from_float(lin, W, s_w, None, fi, bits=bits).to(DEV)
    at = torch.randperm(N, generator=g)[:3 * len(NANS)].to(DEV).view(3, -1)
    for t, where in zip((mod.weights_scales, mod.reduced_w, mod.bias), at):
        t.view(-1)[where] = _bf16(NANS).to(DEV)
    x = torch.randn(M, K + F, generator=g).bfloat16()
    rows = torch.arange(0, M, 97)[:len(NANS)]
    if F:
        x[rows, fi[3]] = _bf16(NANS)[:len(rows)]
    x = x.to(DEV)
    got = mod(x).reshape(M, N).view(torch.int16)
    assert mod._w6 is not None
    nan = torch.zeros(M, N, dtype=torch.bool, device=DEV)
    nan[:, at.reshape(-1)] = True
    if F:
        nan[rows.to(DEV)] = True
    assert torch.equal(got.view(torch.bfloat16).isnan(), nan)
    assert int((got[nan] != 0x7FC0).sum()) == 0
    mod.six_bit_path = False
    assert torch.equal(mod(x).reshape(M, N).view(torch.int16), got)
