"""int8 operand buffers in tile order of more rows than one launch of their quantize kernel takes (2^20): every row as the row-major
operation gives it, which other tests hold against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [1 << 20, (1 << 20) + 1, (1 << 20) + 70])
def test_rows_of_a_further_launch(rows, dtype):
    from quik_amd import asymmetric
    K, F = 64, 32
    fi = np.random.default_rng(rows).permutation(K + F)[:F]
    ii = np.setdiff1d(np.arange(K + F), fi)
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn(rows, K + F, generator=g, device=DEV, dtype=dtype)
    cm = asymmetric.build_colmap(torch.from_numpy(ii).to(DEV), torch.from_numpy(fi).to(DEV), K + F)
    buf, meta8 = asymmetric.quantize_mapped_tile8(x, cm, K, F)
    q, meta, fp_x = asymmetric.quantize_mapped(x, cm, K, F, 8)
    assert torch.equal(meta8.view(torch.int16), meta.view(torch.int16))
    # block of 64 rows, step, half, row of the half, slot (quik_amd/csrc/fp6_format.h): chunk h of a row in slot h ^ (row >> 3 & 1)
    steps = K // 32 + F // 16
    units = buf.view((rows + 63) // 64, steps, 2, 32, 2, 16)
    chunks = torch.empty_like(units)
    swapped = (torch.arange(32, device=DEV) >> 3 & 1).bool()
    chunks[..., ~swapped, :, :], chunks[..., swapped, :, :] = units[..., ~swapped, :, :], units[..., swapped, :, :].flip(-2)
    got = chunks.permute(0, 2, 3, 1, 4, 5).reshape(-1, steps * 32)[:rows]
    assert torch.equal(got[:, :K], q.view(torch.uint8).reshape(rows, K))
    assert torch.equal(got[:, K:], fp_x.contiguous().view(torch.uint8).reshape(rows, 2 * F))
