"""Rounds of a group in the native front end: an override of `finish` is called by every member, members may be called with
other leading sizes than the first, and a finished round leaves nothing behind."""
import pytest
import torch

from test_gpu_front_end import _module, _same

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
N_IN, F, SIZES = 1024 + 64, 64, (256, 64, 72)


def _group(rows):
    from quik_amd.qlinear import SharedQuantizedInput
    shared = SharedQuantizedInput(len(SIZES))
    mods = [_module(i, n, N_IN, F, 4, shared) for i, n in enumerate(SIZES)]
    alone = [_module(i, n, N_IN, F, 4) for i, n in enumerate(SIZES)]
    x = torch.randn(rows, N_IN, generator=torch.Generator().manual_seed(rows)).half().to(DEV)
    want = [a(x)[0] for a in alone]
    for _ in range(2):
        assert all(_same(m(x)[0], w) for m, w in zip(mods, want))
    assert shared._fast is not None
    return shared, mods, x, want


@pytest.mark.parametrize("rows", [6, 36])
def test_leading_sizes_of_a_round(rows):
    shared, mods, x, want = _group(rows)
    shapes = [(rows, N_IN), (1, rows, N_IN), (2, rows // 2, N_IN), (rows, 1, N_IN)]
    for first in shapes:
        for other in shapes:
            for i, (m, w) in enumerate(zip(mods, want)):
                shape = other if i else first
                out = m(x.view(shape))
                lead = shape[:-1] if len(shape) == 3 else (1, rows)
                assert out.shape == (*lead, SIZES[i]) and _same(out.reshape(rows, SIZES[i]), w)
            assert shared.cur_group_elem == 0 and shared._outs is None
    outs = [m(x) for m in mods]          # one round's outputs are their own memory
    for o in outs:
        o.add_(1)
    assert all(_same(m(x)[0], w) for m, w in zip(mods, want))
    assert all(_same(o[0], w + 1) for o, w in zip(outs, want))


@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
def test_an_override_of_finish_is_called(where, monkeypatch):
    from quik_amd.qlinear import SharedQuantizedInput
    shared, mods, x, want = _group(4)
    real, calls = SharedQuantizedInput.finish, []

    def finish(self):
        calls.append(self.cur_group_elem)
        real(self)

    if where == "subclass":
        shared.__class__ = type("Sub", (SharedQuantizedInput,), {"finish": finish})
    elif where == "class":
        monkeypatch.setattr(SharedQuantizedInput, "finish", finish)
    else:
        shared.finish = finish.__get__(shared)
    for n in (1, 2, 3):
        assert all(_same(m(x)[0], w) for m, w in zip(mods, want))
        assert calls == [0, 1, 2] * n and shared._outs is None
