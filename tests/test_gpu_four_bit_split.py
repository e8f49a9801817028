"""K split of the register-streaming tiles on 4-bit weights (csrc/gemm_tile4.hip): which shapes are split, and that a split call
gives the bits of the unsplit one."""
import pytest
import torch

from test_gpu_front_end import _module

DEV = "cuda:0"


def test_what_is_split():
    from quik_amd import _lib as L
    split = L.load().quik_tile4_splitk_bytes
    for shape in ((64, 512, 14336 - 256, 256), (128, 1024, 14336 - 256, 256), (64, 1024, 28672 - 256, 256)):
        assert 4096 < split(*shape) <= 4096 + 256 * 128 * 128 * 4
    # long rows but enough tiles, short rows, many rows
    for shape in ((64, 10240, 8192 - 256, 256), (64, 28672, 8192 - 256, 256), (64, 512, 4096, 0), (2048, 1024, 14336, 0), (0, 512, 14336, 0)):
        assert split(*shape) == 0


# two, three and four workgroups per tile, equal and ragged shares; outlier steps none, some, more than one round of them
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,F,dtype", [(64, 2048, 12288, 0, torch.float16), (40, 4096, 14080, 256, torch.bfloat16),
                                           (33, 1000, 12416, 32, torch.float16), (130, 360, 13056, 544, torch.float16),
                                           (64, 512, 14336, 288, torch.bfloat16), (250, 300, 28544, 96, torch.float16),
                                           (50, 24, 12320, 64, torch.float16)])
def test_split_gives_the_same_bits(M, N, K, F, dtype):
    from quik_amd import _lib as L, matmul
    mod = _module(M, N, K + F, F, 4).to(dtype)
    lib = L.load()
    assert lib.quik_tile4_splitk_bytes(M, N, K, F) > 0 and lib.quik_tile4_activation_bits(M, N, K, F) == 4
    x = torch.randn(M, K + F, generator=torch.Generator().manual_seed(N)).to(dtype).to(DEV)
    got = [mod(x) for _ in range(3)]
    ws = matmul._splitk_workspaces[(torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)]
    assert int(ws[4096:].count_nonzero()) > 0 and int(ws[:4096].view(torch.int32).abs().sum()) == 0
    matmul.split_k = False
    try:
        want = mod(x)
    finally:
        matmul.split_k = True
    for g in got:
        assert torch.equal(g.view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
def test_no_workspace_where_nothing_is_split():
    from quik_amd import matmul
    mod = _module(1, 10240, 8192, 256, 4)
    x = torch.randn(64, 8192, device=DEV).half()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            mod(x)
    side.synchronize()
    assert (torch.cuda.current_device(), side.cuda_stream) not in matmul._splitk_workspaces


@pytest.mark.gpu
def test_a_split_call_in_a_graph():
    """Replayed several times with eager split calls of another input between the replays, on the capture's stream and another."""
    mod = _module(3, 512, 14336, 256, 4)
    g = torch.Generator().manual_seed(0)
    xs = [torch.randn(64, 14336, generator=g).half().to(DEV) for _ in range(4)]
    want = [mod(x).clone() for x in xs]
    held = xs[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = mod(held)
    side = torch.cuda.Stream()
    for i in (1, 2, 3, 0, 2):
        held.copy_(xs[i])
        graph.replay()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            other = mod(xs[3 - i])
        mine = mod(xs[(i + 1) % 4])
        torch.cuda.synchronize()
        for got, k in ((out, i), (other, 3 - i), (mine, (i + 1) % 4)):
            assert torch.equal(got.view(torch.int16), want[k].view(torch.int16))
