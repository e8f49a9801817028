"""The row-major streaming quantize (asym_quantize_stream_kernel) on both sides of the row count up to
which a row of more than 4096 columns gets eight waves (half the CUs), and its persistent form, which prefetches the next row
(int8 operand buffers of more fp16 rows than CUs, beyond 16384 columns, that the ring kernel does not take), with workgroups that take
more than one row.  bf16 rows of that length take quantize_units_kernel.  Against the oracle."""
import numpy as np
import pytest
import torch

from oracle import quik_oracle as qo
from test_gpu_long_row_quantize import decode_tile8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _few():
    return torch.cuda.get_device_properties(0).multi_processor_count // 2


def _case(rows, n_in, fi, bf16, seed):
    rng = np.random.default_rng(seed)
    ii = np.setdiff1d(np.arange(n_in), fi).astype(np.int64)
    x = rng.standard_normal((rows, n_in), dtype=np.float32)
    x[:, fi] *= 50
    x[0, :], x[rows - 1, ii[0]], x[rows - 1, ii[-1]] = 1.5, np.nan, 300.0
    x[rows // 2, ii[3]], x[rows // 2, ii[4]] = (3e38, -3e38) if bf16 else (65504.0, -65504.0)
    if bf16:
        x = qo.bf16_round(x)
        return x, torch.from_numpy(x).bfloat16().to(DEV), ii
    x = x.astype(np.float16)
    return x, _t(x), ii


def _bits(t):
    return t.cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _patterns(a, bf16):
    return qo.f32_to_bf16_bits(a) if bf16 else a.view(np.uint16)


def _check_meta(meta, want, bf16):
    got, bits = _bits(meta).reshape(-1, 2), _patterns(want, bf16).reshape(-1, 2)
    zero = np.asarray(want, np.float32).reshape(-1, 2)[:, 1]
    assert np.array_equal(got[:, 0], bits[:, 0])
    assert np.array_equal(meta.float().cpu().numpy().reshape(-1, 2)[:, 1], zero, equal_nan=True)


@pytest.mark.parametrize("beyond", [0, 1])
@pytest.mark.parametrize("n_in,F", [(4104, 40), (8192, 256), (12288, 700), (16392, 64)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("bf16", [False, True])
def test_eight_waves_per_row_or_four(beyond, n_in, F, bits, bf16):
    from quik_amd import asymmetric
    rows = _few() + beyond
    fi = np.random.default_rng(n_in).permutation(n_in)[:F].astype(np.int64)
    x, xt, ii = _case(rows, n_in, fi, bf16, n_in + bits)
    cm = asymmetric.build_colmap(_t(ii), _t(fi), n_in)
    assert asymmetric.colmap_streams(cm, n_in - F, F)
    q, meta, fp_x = asymmetric.quantize_mapped(xt, cm, n_in - F, F, bits)
    with np.errstate(all="ignore"):
        want_q, want_meta, want_fp = qo.asym_quantize(x, ii, fi, bits, *([qo.BF16] if bf16 else []))
    assert np.array_equal(q.cpu().numpy(), want_q)
    assert np.array_equal(_bits(fp_x).reshape(rows, F), _patterns(want_fp, bf16).reshape(rows, F))
    _check_meta(meta, want_meta, bf16)


@pytest.mark.parametrize("beyond", [0, 1])
@pytest.mark.parametrize("n_in,F", [(4104, 40), (8192, 256), (16392, 64)])
@pytest.mark.parametrize("bits", [4, 8])
def test_eight_waves_per_row_or_four_symmetric(beyond, n_in, F, bits):
    from quik_amd import symmetric
    from quik_amd.asymmetric import build_colmap
    rows, divisor = _few() + beyond, 7.0 if bits == 4 else 127.0
    fi = np.random.default_rng(n_in).permutation(n_in)[:F].astype(np.int64)
    ii = np.setdiff1d(np.arange(n_in), fi).astype(np.int64)
    g = torch.Generator().manual_seed(n_in + bits)
    x = torch.randn(rows, n_in, generator=g)
    x[:, fi] *= 50
    x = x.half().to(DEV)
    q, scale, fp_x = symmetric.quantize_mapped(x, build_colmap(_t(ii), _t(fi), n_in), n_in - F, F, bits, divisor, False)
    int_x = x[:, _t(ii)].contiguous()
    want = (int_x.abs().max(dim=1)[0].unsqueeze(1) / divisor).half()
    assert torch.equal(scale, want)
    assert torch.equal(q, symmetric.quantize(int_x, want, bits))
    assert torch.equal(fp_x, x[:, _t(fi)])


@pytest.mark.parametrize("rows,n_in,F,bf16", [(300, 28672, 256, True), (700, 16512, 128, True), (1100, 16416, 32, True),
                                              (600, 20480, 1024, False), (530, 32768, 256, False)])
def test_persistent_workgroups(rows, n_in, F, bf16):
    """bf16 rows (a workgroup each), fp16 rows with an outlier column in each of more groups than the ring kernel takes, fp16 rows
    beyond what its ring holds; two workgroups per CU, so more than 512 rows are more than one row for some of them."""
    from quik_amd import asymmetric
    rng = np.random.default_rng(rows)
    fi = (np.arange(F) * 8 + rng.integers(0, 8, F) if F == 1024 else rng.permutation(n_in)[:F]).astype(np.int64)
    x, xt, ii = _case(rows, n_in, fi, bf16, rows + F)
    K = n_in - F
    cm = asymmetric.build_colmap(_t(ii), _t(fi), n_in)
    assert asymmetric.colmap_streams(cm, K, F)
    x8, meta = asymmetric.quantize_mapped_tile8(xt, cm, K, F)
    with np.errstate(all="ignore"):
        want_q, want_meta, want_fp = qo.asym_quantize(x, ii, fi, 8, *([qo.BF16] if bf16 else []))
    codes, outl = decode_tile8(x8.cpu().numpy(), rows, K, F)
    assert np.array_equal(codes, want_q)
    assert np.array_equal(outl, _patterns(want_fp, bf16).reshape(rows, F))
    _check_meta(meta, want_meta, bf16)
