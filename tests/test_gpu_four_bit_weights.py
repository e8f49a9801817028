"""4-bit weights in tile order: the buffers hold the codes (layout restated from quik_amd/csrc/fp6_format.h), and the GEMMs on
them, activation in 4 or in 6 bits, give the bits of the 6-bit path, which the oracle pins."""
import numpy as np
import pytest
import torch

from test_gpu_parity import _bits, _decode_operand6, _in_place_order, _t

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _to_six_bit_buffer(buf, rows, K, F):
    """A 4-bit operand buffer as the 6-bit buffer of the same levels (K a multiple of 128)."""
    units, blocks = K // 64 + F // 16, (rows + 63) // 64
    u = buf[:blocks * units * 2048].reshape(blocks, units, 2, 32, 2, 16)      # half, row, slot
    out = np.zeros((blocks, units, 3072), np.uint8)
    out[:, :, :2048] = u.reshape(blocks, units, 2048)
    p = u[:, :K // 64].copy().view(np.uint32).astype(np.uint64)               # [block, step, half, row, slot, 4]
    fields = np.zeros(p.shape[:-1] + (32,), np.uint64)
    for part in range(2):
        p0, p1 = p[..., 2 * part], p[..., 2 * part + 1]
        for e in range(16):
            at = 6 * e
            if e < 5:
                f = p0 >> np.uint64(at) & np.uint64(15)
            elif e == 5:
                f = p0 >> np.uint64(30) | (p1 & np.uint64(3)) << np.uint64(2)
            elif e < 11:
                f = p1 >> np.uint64(at - 32) & np.uint64(15)
            else:
                f = (p1 >> np.uint64(at - 64) & np.uint64(3)) | (p0 >> np.uint64(at - 64) & np.uint64(12))
            fields[..., 16 * part + e] = f
    for slot in range(2):
        for half in range(2):
            for r in range(32):
                h, row = slot ^ ((r >> 3) & 1), half * 32 + r
                f = fields[:, :, half, r, slot]
                word = np.zeros(f.shape[:2] + (192,), np.uint8)
                for e in range(32):
                    for b in range(4):
                        word[..., 6 * e + b] = f[..., e] >> np.uint64(b) & np.uint64(1)
                packed = np.packbits(word, axis=-1, bitorder="little")
                out[:, :K // 64, half * 1024 + r * 32 + slot * 16:][..., :16] = packed[..., :16]
                out[:, :K // 64, 2048 + h * 512 + row * 8:][..., :8] = packed[..., 16:]
    return np.concatenate([out.reshape(-1), buf[blocks * units * 2048:][:4 * rows]])


def _problem(M, N, K, F, seed, dtype=torch.float16):
    from quik_amd import asymmetric
    g = torch.Generator(device=DEV).manual_seed(seed)
    n_in = K + F
    fi = torch.randperm(n_in, generator=g, device=DEV)[:F]
    keep = torch.ones(n_in, dtype=torch.bool, device=DEV)
    keep[fi] = False
    ii = torch.arange(n_in, device=DEV)[keep]
    x = torch.randn(M, n_in, generator=g, device=DEV)
    x[:, fi] *= 50
    qw = torch.randint(0, 256, (N, K // 2), generator=g, device=DEV, dtype=torch.int16).to(torch.uint8)
    fw = (0.02 * torch.randn(N, F, generator=g, device=DEV)).to(dtype)
    return ii, fi, asymmetric.build_colmap(ii, fi, n_in), x.to(dtype), qw, fw, g


@pytest.mark.parametrize("rows,K,F,kind", [(1, 128, 0, "fp16"), (70, 256, 32, "fp16"), (130, 384, 96, "bf16"), (33, 256, 64, "symmetric"),
                                           (9, 16384 + 256, 160, "fp16")])
def test_buffers_hold_the_codes(rows, K, F, kind):
    from quik_amd import asymmetric, matmul, symmetric
    ii, fi, cm, x, qw, fw, _ = _problem(rows, rows, K, F, rows + K, torch.bfloat16 if kind == "bf16" else torch.float16)
    x[rows - 1, ii[0]], x[rows - 1, ii[-1]] = float("nan"), 300.0
    if kind == "symmetric":
        x4, meta4 = symmetric.quantize_mapped(x, cm, K, F, 4, 4, True, True)[:2]
        q, meta, fp_x = symmetric.quantize_mapped(x, cm, K, F, 4, 4, False)
    else:
        x4, meta4 = asymmetric.quantize_mapped_fp6(x, cm, K, F, True)
        q, meta, fp_x = asymmetric.quantize_mapped(x, cm, K, F, 4)
    assert np.array_equal(_bits(meta), _bits(meta4))
    order = _in_place_order(ii.cpu().numpy(), fi.cpu().numpy(), K + F)
    for buf, codes, outliers in ((x4, q, fp_x), (matmul.pack_weight_fp6(qw, fw, cm, True), qw, fw)):
        c = codes.cpu().numpy()
        want = np.empty((rows, K), np.int64)
        want[:, 0::2], want[:, 1::2] = (c & 0xF) ^ 8, (c >> 4) ^ 8
        levels, outl, sums = _decode_operand6(_to_six_bit_buffer(buf.cpu().numpy(), rows, K, F), rows, K, F)
        assert np.array_equal(levels, want[:, order])
        assert np.array_equal(outl, _bits(outliers).reshape(rows, F) if F else outl)
        assert np.array_equal(sums, want.sum(1))


# every kernel: 64x32, 64x64 and 128x64 tiles (steps of a wave below, at and beyond what it keeps in flight; outlier steps none,
# in one round, in several; ragged edges; more tiles than CUs), 128x128, 256x256 and 256x128 tiles, a rest behind whole rounds
SHAPES = [(1, 8, 128, 0), (33, 40, 128, 32), (64, 32, 1024, 0), (63, 100, 2048, 64), (65, 1000, 2176, 256), (64, 4096, 3840, 288),
          (200, 2048 + 24, 4224, 512), (64, 10240, 7936, 256), (130, 8192, 896, 32), (300, 4544, 4096 + 256, 128),
          (257, 7000, 1152, 96), (2048, 1024, 640, 512), (777, 4096, 1920, 64), (1000, 5000, 1024, 320), (777, 11008, 512, 32),
          (2048, 8192, 256, 0), (2048, 9216, 384, 64), (1300, 13824 + 8, 256, 32)]


@pytest.mark.parametrize("M,N,K,F", SHAPES)
def test_gemm_gives_the_bits_of_the_six_bit_path(M, N, K, F):
    from quik_amd import asymmetric, matmul, symmetric
    bf16, symm, bias = (M + N) % 3 == 0, (M + N) % 3 == 1, (M + K // 128) % 2 == 0
    dtype = torch.bfloat16 if bf16 else torch.float16
    _, _, cm, x, qw, fw, g = _problem(M, N, K, F, M + N + K, dtype)
    s_col = (torch.rand(N, 1, generator=g, device=DEV) * 0.009 + 0.001).to(dtype)
    wr = None if symm else torch.randn(1, N, generator=g, device=DEV).to(dtype)
    b = torch.randn(N, generator=g, device=DEV).to(dtype) if bias else None

    def quantize(four):
        if symm:
            return symmetric.quantize_mapped(x, cm, K, F, 4, 4, True, four)[:2]
        return asymmetric.quantize_mapped_fp6(x, cm, K, F, four)
    x6, meta = quantize(False)
    x4, _ = quantize(True)
    want = matmul.mixed_linear_fp6(x6, matmul.pack_weight_fp6(qw, fw, cm), meta, s_col, wr, b, M, N, K, F, dtype)
    w4 = matmul.pack_weight_fp6(qw, fw, cm, True)
    for xb in (x4, x6):
        got = matmul.mixed_linear_tile4(xb, w4, meta, s_col, wr, b, M, N, K, F, dtype)
        assert np.array_equal(_bits(got), _bits(want)), xb.numel()


@pytest.mark.parametrize("M,N,n_in,F", [(33, 520, 160, 0), (64, 300, 992, 32), (300, 1096, 4544, 128), (2048, 2304, 736, 64)])
def test_layer_whose_columns_do_not_fill_the_steps(M, N, n_in, F):
    """The last k-steps are filled up: against the row-major kernels."""
    from quik_amd.qlinear import MixedQLinear
    K = n_in - F
    ii, fi, _, x, qw, fw, g = _problem(M, N, K, F, N, torch.float16)
    mods = []
    for path in (True, False):
        m = MixedQLinear(n_in, N, None, fp_features_num=F, bits=4).to(DEV)
        m.int_indices, m.fp_indices, m.int_weight = ii, fi, qw
        if F:
            m.fp_weight = fw
        m.weights_scales = (torch.rand(N, 1, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV) * 0.01).half()
        m.reduced_w = torch.linspace(-1, 1, N, device=DEV).half()[None]
        m.six_bit_path = path
        mods.append(m)
    a, b = mods[0](x), mods[1](x)
    assert mods[0]._w6_four and mods[1]._w6 is None
    assert np.array_equal(_bits(a), _bits(b))
