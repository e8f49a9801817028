"""The 6-bit operand output of the quantize (quantize_fp6_row_kernel, a workgroup per row) against the codes of the row-major
quantize, which the oracle pins: one wave and eight, one fragment per lane and two (beyond 16384 columns), rows that end
inside a wave, more holes and outlier chunks than lanes, row counts that leave places without a row.  Same bits."""
import numpy as np
import pytest
import torch

from test_gpu_parity import _bits, _decode_operand6, _in_place_order, _t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,K,F", [(1, 128, 0), (9, 128, 32), (3, 1920, 96), (5, 2048, 32), (8, 1024, 1024), (17, 256, 1760),
                                      (2, 4096, 4096), (7, 16384 - 256, 256), (3, 16384 - 128, 160), (2, 32768 - 512, 480),
                                      (2, 16384, 16384), (1025, 2304, 32)])
@pytest.mark.parametrize("kind", ["fp16", "bf16", "symmetric"])
def test_levels_outliers_and_sums(rows, K, F, kind):
    from quik_amd import asymmetric, symmetric
    n_in = K + F
    rng = np.random.default_rng(rows + K + F)
    perm = rng.permutation(n_in)
    fi, ii = perm[:F].astype(np.int64), np.sort(perm[F:]).astype(np.int64)
    x = rng.standard_normal((rows, n_in)).astype(np.float32)
    x[:, fi] *= 50
    x[rows - 1, ii[0]], x[rows - 1, ii[-1]] = np.nan, 300.0
    xt = torch.from_numpy(x).to("cuda:0").to(torch.bfloat16 if kind == "bf16" else torch.float16)
    if rows > 2 and kind != "symmetric":
        xt[1] = 6e4 * torch.sign(xt[1])            # a range beyond what fp16 holds
    cm = asymmetric.build_colmap(_t(ii), _t(fi), n_in)
    assert asymmetric.colmap_streams(cm, K, F)
    if kind == "symmetric":
        x6, meta6 = symmetric.quantize_mapped(xt, cm, K, F, 4, 4, True)[:2]
        q, meta, fp_x = symmetric.quantize_mapped(xt, cm, K, F, 4, 4, False)
    else:
        x6, meta6 = asymmetric.quantize_mapped_fp6(xt, cm, K, F)
        q, meta, fp_x = asymmetric.quantize_mapped(xt, cm, K, F, 4)
    assert np.array_equal(_bits(meta), _bits(meta6))
    qn = q.cpu().numpy()
    want = np.empty((rows, K), np.int64)
    want[:, 0::2], want[:, 1::2] = (qn & 0xF) ^ 8, (qn >> 4) ^ 8
    levels, outl, sums = _decode_operand6(x6.cpu().numpy(), rows, K, F)
    assert np.array_equal(levels, want[:, _in_place_order(ii, fi, n_in)])
    assert np.array_equal(outl, _bits(fp_x).reshape(rows, F) if F else outl)
    assert np.array_equal(sums, want.sum(1))
