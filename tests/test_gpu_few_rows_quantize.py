"""Quantize of a layer's few rows (quantize_units_kernel in csrc/quantize.hip): codes, scales, zero points and outlier values of a
forward's workspace, bit for bit those of the stand-alone operation, which other tests hold against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_one_launch_decode import _call, _layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# rows, K, F, bits, outlier columns in runs: one, two, four and eight groups of eight columns per lane and their ends, more outlier columns than
# lanes, none, rows of less than a kilobyte; more gathered units than lanes; the last is left to the other kernel (more rows)
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


# (rows: up to and beyond those of fp16 rows of more than 16384 columns)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,K,F,runs", [(1, 64, 32, False), (33, 480, 32, True), (65, 4096, 32, False), (130, 4064, 0, False), (40, 8192, 32, True),
                                           (257, 7952, 256, False), (70, 16128, 256, True), (300, 16384, 32, False), (256, 16512, 128, False),
                                           (257, 16512, 128, False), (35, 32512, 256, False), (9, 31744, 1024, False)])
def test_tile_order_holds_what_the_operation_gives(rows, K, F, runs, dtype):
    """The buffer's chunks (layout restated from quik_amd/csrc/fp6_format.h) against the codes and values in row order."""
    from quik_amd import asymmetric
    rng = np.random.default_rng(K + F + rows)
    mod, _, _, fi, ii, _ = _layer(rng, 16, K + F, F, 8, dtype, runs)
    x = rng.standard_normal((rows, K + F)).astype(np.float32)
    x[:, fi] *= 50
    x[0, ii[3]], x[rows // 2, ii[0]], x[rows // 2, ii[-1]] = np.nan, 6e4, -6e4
    x[rows - 1, ii[K // 2]] = np.inf
    xt = torch.from_numpy(x).to(DEV, dtype)
    q, meta, fp_x = asymmetric.quantize_mapped(xt, mod._column_map(), K, F, 8)
    buf, meta8 = asymmetric.quantize_mapped_tile8(xt, mod._column_map(), K, F) if K % 64 == 0 else _through_the_layer(mod, xt)
    assert torch.equal(meta8.view(torch.int16)[:2 * rows], meta.view(torch.int16))
    steps, r = (K + 63) // 64 * 2, torch.arange(rows, device=DEV)
    units = buf[:(rows + 63) // 64 * (steps + F // 16) * 2048].view(-1, steps + F // 16, 2, 32, 2, 16)   # block, step, half, row, slot
    swap = (r >> 3) & 1
    for want, first in ((q.view(torch.uint8), 0), (fp_x.contiguous().view(torch.uint8).reshape(rows, -1), steps)):
        chunks = want.shape[1] // 16
        c = torch.arange(chunks, device=DEV)
        got = units[(r >> 6)[:, None], first + (c >> 1)[None], ((r >> 5) & 1)[:, None], (r & 31)[:, None], (c & 1)[None] ^ swap[:, None]]
        assert torch.equal(got.reshape(rows, -1), want)


def _through_the_layer(mod, xt):
    """Operand buffer and scales in the workspace of a forward on the tile-ordered path."""
    import ctypes
    from quik_amd import _lib as L
    lib, rows = L.load(), xt.shape[0]
    desc, _ = mod._descriptor(True)
    n = lib.quik_layer_workspace_bytes(ctypes.byref(desc), rows)
    ws, out = torch.zeros(n, dtype=torch.uint8, device=DEV), torch.empty(rows, mod.out_features, dtype=xt.dtype, device=DEV)
    L.check(lib.quik_layer_forward(ctypes.byref(desc), xt.data_ptr(), rows, ws.data_ptr(), n, None, 0, out.data_ptr(), None, L.stream()), "forward")
    K, F = mod.int_features_num, mod.fp_features_num
    at = ((rows + 63) // 64 * ((K + 63) // 64 * 2 + F // 16) * 2048 + 255) // 256 * 256
    return ws, ws[at:at + 4 * rows].view(xt.dtype)


@pytest.mark.parametrize("bits", [4, 8])
def test_a_few_rows_take_the_map_that_is_there(bits):
    """A captured forward whose layer's map is another one at its replays: one with more gathered units, one that does not stream."""
    from quik_amd import asymmetric
    rows, K, F = 5, 1024, 64
    rng = np.random.default_rng(0)
    mod, _, _, fi, _, _ = _layer(rng, 16, K + F, F, bits, torch.float16, False)
    x = torch.randn(rows, K + F, device=DEV).half()
    orders = [(np.arange(K), np.arange(K, K + F))]                                     # no gathered unit
    out = rng.permutation(K + F)[:F]
    orders.append((np.setdiff1d(np.arange(K + F), out), out))                          # many
    orders.append((orders[1][0][::-1].copy(), out))                                    # no ascending order
    maps = [asymmetric.build_colmap(torch.from_numpy(i).to(DEV), torch.from_numpy(f).to(DEV), K + F) for i, f in orders]
    cm = mod._column_map()
    cm.copy_(maps[0])
    mod(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = mod(x)
    for k in (1, 2, 0, 1):
        cm.copy_(maps[k])
        graph.replay()
        q, meta, fp_x = asymmetric.quantize_mapped(x, maps[k], K, F, bits)
        from quik_amd import matmul
        acc = (matmul.int4Matmul if bits == 4 else matmul.int8Matmul)(q, mod.int_weight)
        z = torch.nn.functional.linear(fp_x, mod.fp_weight)
        want = asymmetric.dequantize(acc, meta, mod.weights_scales, mod.reduced_w, z, bits).float() + mod.bias.float()
        rms = want.pow(2).mean().sqrt()
        assert (y.float() - want).abs().max() <= 1e-2 * rms, k   # (16-bit outlier products and results, as the fused forward's tests)


@pytest.mark.parametrize("K,F,bits,runs", [c[1:] for c in CASES])
def test_symmetric_few_rows(K, F, bits, runs):
    """Few rows of symmetric activations against the same rows in a call of more, which the streaming kernel takes: bit for bit."""
    from quik_amd import symmetric
    rng = np.random.default_rng(K + F)
    mod, _, _, fi, ii, _ = _layer(rng, 16, K + F, F, bits, torch.float16, runs)
    x = rng.standard_normal((40, K + F)).astype(np.float32)
    x[:, fi] *= 50
    x[0, ii[3]], x[1, ii[K // 2]], x[2], x[3, ii[-1]], x[4] = np.nan, -np.inf, 0, -6e4, 1e-7
    xt = torch.from_numpy(x).to(DEV, torch.float16)
    if F:
        xt[5, fi] = float("nan")
    cm, divisor = mod._column_map(), 7.0 if bits == 4 else 127.0
    want = symmetric.quantize_mapped(xt, cm, K, F, bits, divisor, False)
    for rows in (1, 7, 32):
        got = symmetric.quantize_mapped(xt[:rows], cm, K, F, bits, divisor, False)
        for g, w in zip(got, want):
            if g is not None:
                assert torch.equal(g.contiguous().view(torch.uint8), w[:rows].contiguous().view(torch.uint8))
