"""The native front end (csrc/front.cpp) behind MixedQLinear.forward and the stand-alone operations.

A repeated forward runs through a plan made by the first one; whatever the plan was made from may change between two
calls (a buffer written in place or replaced, a switch of the module or of its class, the input's form), and the
next call has to see it.  Every check compares bits with a module built afresh in the changed state.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _module(seed, N, n_in, F, bits, shared=None, bias=False, outlier_seed=1):
    from quik_amd.qlinear import MixedQLinear
    rng = np.random.default_rng(seed)
    fi = torch.from_numpy(np.sort(np.random.default_rng(outlier_seed).permutation(n_in)[:F]))
    s_w = torch.from_numpy(rng.uniform(0.001, 0.01, (N, 1)).astype(np.float16))
    lo, hi = (-8, 8) if bits == 4 else (-127, 128)
    W = torch.from_numpy((rng.integers(lo, hi, (N, n_in)) * s_w.float().numpy()).astype(np.float16))
    lin = torch.nn.Linear(n_in, N, bias=bias, dtype=torch.float16)
    if bias:
        lin.bias.data = torch.from_numpy(rng.standard_normal(N).astype(np.float16))
    return MixedQLinear.from_float(lin, W, s_w, shared, fi, bits=bits).to(DEV)


def _same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def _planned(mod):
    return "fast" in mod._descs


@pytest.mark.parametrize("rows", [1, 2, 3, 32, 33, 70])
@pytest.mark.parametrize("bits", [4, 8])
def test_a_planned_forward_sees_every_change(rows, bits):
    from quik_amd.qlinear import MixedQLinear
    N, n_in, F = 264, 1024 + 64, 64
    mod = _module(0, N, n_in, F, bits, bias=True)
    x = torch.randn(rows, n_in, generator=torch.Generator().manual_seed(rows)).half().to(DEV)
    first = mod(x)
    assert _planned(mod)
    assert _same(mod(x), first) and mod(x).shape == (1, rows, N)
    assert mod(x[None]).shape == (1, rows, N)
    # a form the plan does not take: a view with other strides, another type of tensor
    wide = torch.zeros(rows, 2 * n_in, dtype=torch.float16, device=DEV)
    wide[:, :n_in] = x
    assert _same(mod(wide[:, :n_in]), first)
    assert _same(mod(torch.nn.Parameter(x, requires_grad=False)), first)
    with pytest.raises(RuntimeError):
        mod(x[:, :-1].contiguous())
    # in place, replaced, and back
    other = _module(7, N, n_in, F, bits, bias=True)
    mod.load_state_dict(other.state_dict())
    want = other(x)
    assert not _same(want, first)
    assert _same(mod(x), want) and _same(mod(x), want)
    mod.bias = None
    no_bias = _module(7, N, n_in, F, bits)
    assert _same(mod(x), no_bias(x)) and _same(mod(x), no_bias(x))
    mod.weights_scales.data = mod.weights_scales.data * 2      # (a new address, no new version of the old tensor)
    no_bias.weights_scales.mul_(2)
    assert _same(mod(x), no_bias(x))
    # switches of the module and of the class
    mod.six_bit_path = False
    assert _same(mod(x), no_bias(x)) or rows <= 32
    keep = MixedQLinear.six_bit_min_rows
    calls = []
    real = MixedQLinear._forward_one_call
    try:
        MixedQLinear._forward_one_call = lambda self, x2: calls.append(1) or real(self, x2)
        for n in (1, 2, 3):
            mod(x)
            assert calls == [1] * n
    finally:
        MixedQLinear._forward_one_call = real
    assert MixedQLinear.six_bit_min_rows == keep


def _rewrite(mod, other):
    mod.load_state_dict(other.state_dict())


def _assign(mod, other):
    mod.load_state_dict({k: v.clone() for k, v in other.state_dict().items()}, assign=True)


def _move(mod, other):
    mod.cpu()
    mod.load_state_dict(other.state_dict())
    mod.to(DEV)


def _offload(mod, other):                                  # (the blocks given back are handed out again)
    for name, b in mod.named_buffers():
        b.data = b.data.cpu()
    for name, b in mod.named_buffers():
        b.data.copy_(getattr(other, name))
        b.data = b.data.to(DEV)


@pytest.mark.parametrize("change", [_rewrite, _assign, _move, _offload])
@pytest.mark.parametrize("outliers", [1, 2])               # the same outlier columns as before, or others
@pytest.mark.parametrize("before,after", [((64, 1), (1, 64)), ((1, 64), (64, 1)), ((64, 1), (64, 1)), ((64,), (1, 64))])
@pytest.mark.parametrize("bits", [4, 8])
def test_both_paths_see_a_change_of_the_weights(bits, before, after, outliers, change):
    N, n_in, F = 264, 1024 + 64, 64
    mod, other = (_module(s, N, n_in, F, bits, bias=True, outlier_seed=o) for s, o in ((0, 1), (7, outliers)))
    xs = {r: torch.randn(r, n_in, generator=torch.Generator().manual_seed(r)).half().to(DEV) for r in (1, 64)}
    for rows in before + before:
        mod(xs[rows])
    change(mod, other)
    for rows in after + after:
        assert _same(mod(xs[rows]), other(xs[rows]))


def test_a_plan_keeps_no_weights_alive():
    mod = _module(0, 4096, 4096 + 64, 64, 4)
    x = torch.randn(1, 4096 + 64, generator=torch.Generator().manual_seed(0)).half().to(DEV)
    mod(x)
    assert _planned(mod)
    before, held = torch.cuda.memory_allocated(), mod.weight_bytes()["row_major"]
    mod.cpu()
    assert before - torch.cuda.memory_allocated() >= held


@pytest.mark.parametrize("bits", [4, 8])
def test_transient_policy_set_after_a_prefill(bits):
    N, n_in, F = 264, 1024 + 64, 64
    mod, other = _module(0, N, n_in, F, bits), _module(7, N, n_in, F, bits)
    xs = {r: torch.randn(r, n_in, generator=torch.Generator().manual_seed(r)).half().to(DEV) for r in (1, 64)}
    for rows in (64, 1, 64):
        mod(xs[rows])
    mod.transient_tiled_copy = True
    for rows in (64, 1, 64):
        mod(xs[rows])
        assert mod.weight_bytes()["tiled"] == 0
    mod.load_state_dict(other.state_dict())
    for rows in (64, 1, 64, 64):
        assert _same(mod(xs[rows]), other(xs[rows]))


def test_a_call_that_goes_back_keeps_its_event():
    N, n_in, rows = 16384, 1024, 8192
    mod = _module(0, N, n_in, 0, 4)
    x = torch.zeros(rows, n_in, dtype=torch.float16, device=DEV)
    mod(x[:64])
    assert _planned(mod)
    event = torch.cuda.Event()
    event.record()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:                                                   # no room for the 256 MB result
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
        mod.mid_event = event
        with pytest.raises(torch.OutOfMemoryError):
            mod(x)
        assert mod.mid_event is event and _planned(mod)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    mod(x)
    assert mod.mid_event is None
    torch.cuda.synchronize()
    assert event.query()


@pytest.mark.parametrize("rows", [1, 40])
def test_a_planned_group_sees_every_change(rows):
    from quik_amd.qlinear import SharedQuantizedInput
    n_in, F, sizes = 1024 + 64, 64, (256, 64, 64)
    shared = SharedQuantizedInput(3)
    mods = [_module(i, n, n_in, F, 4, shared) for i, n in enumerate(sizes)]
    alone = [_module(i, n, n_in, F, 4) for i, n in enumerate(sizes)]
    x = torch.randn(rows, n_in, generator=torch.Generator().manual_seed(3)).half().to(DEV)
    for _ in range(3):
        for m, a in zip(mods, alone):
            assert _same(m(x), a(x))
        assert shared._fast is not None and shared.cur_group_elem == 0 and shared._outs is None
    for order in ((2, 0, 1), (1, 2, 0)):                     # any call order
        for i in order:
            assert _same(mods[i](x[None]), alone[i](x[None]))
    for m, a in zip(mods, alone):                            # one member's scales change in place
        m.weights_scales.mul_(2)
        a.weights_scales.mul_(2)
    for _ in range(2):
        for m, a in zip(mods, alone):
            assert _same(m(x), a(x))
    outs = [mods[0](x)]                                      # a switch set in the middle of a round
    mods[1].fuse_shared_groups = True
    outs += [mods[1](x), mods[2](x)]
    assert all(_same(o, a(x)) for o, a in zip(outs, alone))
    assert shared.cur_group_elem == 0


@pytest.mark.parametrize("name", ["int_weight", "weights_scales", "fp_weight", "reduced_w", "bias"])
@pytest.mark.parametrize("change", [_rewrite, _assign])
def test_both_paths_of_a_group_see_a_change_of_one_buffer(change, name):
    from quik_amd.qlinear import SharedQuantizedInput
    n_in, F, sizes = 1024 + 64, 64, (256, 64)
    xs = {r: torch.randn(r, n_in, generator=torch.Generator().manual_seed(r)).half().to(DEV) for r in (1, 64)}
    for before, after in (((64, 1), (1, 64)), ((1, 64), (64, 1)), ((64, 1), (64, 1))):
        shared = SharedQuantizedInput(2)
        mods = [_module(i, n, n_in, F, 4, shared, bias=True) for i, n in enumerate(sizes)]
        alone = [_module(i, n, n_in, F, 4, bias=True) for i, n in enumerate(sizes)]
        for rows in before + before:
            for m in mods:
                m(xs[rows])
        assert shared._fast is not None
        new = {name: getattr(_module(9, sizes[1], n_in, F, 4, bias=True), name)}
        if change is _rewrite:
            mods[1].load_state_dict(new, strict=False)
        else:
            mods[1].load_state_dict({name: new[name].clone()}, strict=False, assign=True)
        alone[1].load_state_dict(new, strict=False)
        for rows in after + after:
            for m, a in zip(mods, alone):
                assert _same(m(xs[rows]), a(xs[rows]))
            assert shared._fast is not None


@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
def test_an_override_of_the_group_is_called_by_every_round(where, monkeypatch):
    from quik_amd.qlinear import SharedQuantizedInput
    n_in, F, sizes, calls = 1024 + 64, 64, (256, 64), []
    real = SharedQuantizedInput.group_forward

    def override(self, *args):
        calls.append(1)
        return real(self, *args)

    x = torch.randn(1, n_in, generator=torch.Generator().manual_seed(0)).half().to(DEV)
    shared = SharedQuantizedInput(2)
    mods = [_module(i, n, n_in, F, 4, shared) for i, n in enumerate(sizes)]
    first = [m(x) for m in mods]
    assert shared._fast is not None and all(_same(m(x), f) for m, f in zip(mods, first))
    if where == "subclass":
        shared.__class__ = type("Sub", (SharedQuantizedInput,), {"group_forward": override})
    elif where == "class":
        monkeypatch.setattr(SharedQuantizedInput, "group_forward", override)
    else:
        shared.group_forward = override.__get__(shared)
    for n in (1, 2, 3):
        assert all(_same(m(x), f) for m, f in zip(mods, first))
        assert len(calls) == 2 * n


def test_a_switch_of_one_member_is_seen():
    from quik_amd.qlinear import SharedQuantizedInput
    n_in, F, sizes = 1024 + 64, 64, (256, 64)
    x = torch.randn(64, n_in, generator=torch.Generator().manual_seed(0)).half().to(DEV)
    shared = SharedQuantizedInput(2)
    mods = [_module(i, n, n_in, F, 4, shared) for i, n in enumerate(sizes)]
    alone = [_module(i, n, n_in, F, 4) for i, n in enumerate(sizes)]
    for switch in (None, "fused", "fuse_shared_groups"):
        if switch is not None:
            for m in (mods[1], alone[1]):
                setattr(m, switch, False)
        for _ in range(2):
            assert all(_same(m(x), a(x)) for m, a in zip(mods, alone))
        assert switch is None or "fast" not in mods[1]._descs
        for m in (mods[1], alone[1]):
            m.fused = m.fuse_shared_groups = True


def test_same_bits_without_the_front_end(monkeypatch):
    import quik
    from quik_amd import _lib as L
    mod = _module(0, 264, 1024 + 64, 64, 4)
    xs = [torch.randn(r, 1024 + 64, generator=torch.Generator().manual_seed(r)).half().to(DEV) for r in (1, 64)]

    def ops(x):
        q, meta, fp_x = quik.asymmetric.quantize(x, mod.int_indices, mod.fp_indices, 4)
        acc = quik.matmul.int4Matmul(q, mod.int_weight)
        y = torch.nn.functional.linear(fp_x, mod.fp_weight)
        return [q, meta, fp_x, acc, quik.asymmetric.dequantize(acc, meta, mod.weights_scales, mod.reduced_w, y, 4)]
    want = [(mod(x), ops(x)) for x in xs]
    assert _planned(mod)
    monkeypatch.setattr(L, "_front", L._NoFront())
    bare = _module(0, 264, 1024 + 64, 64, 4)
    for x, (out, parts) in zip(xs, want):
        for _ in range(2):
            assert _same(bare(x), out) and not _planned(bare)
        assert all(torch.equal(a, b) for a, b in zip(ops(x), parts))


def test_interposed_inputs_stay_with_the_python_functions():
    from torch.utils._python_dispatch import TorchDispatchMode
    import quik
    mod = _module(0, 256, 1024, 0, 4)
    x = torch.randn(4, 1024, generator=torch.Generator().manual_seed(0)).half().to(DEV)
    first = mod(x)
    assert _planned(mod)
    ii, fi = mod.int_indices, mod.fp_indices
    for call in (mod, lambda t: quik.asymmetric.quantize(t, ii, fi, 4)[0]):
        # a level's tensor has no memory to hand to a kernel: the error of its data pointer, not an abort
        with pytest.raises(RuntimeError):
            torch.vmap(call)(x[None])
        with pytest.raises(RuntimeError):
            torch.func.jvp(call, (x,), (x,))

    class Seen(TorchDispatchMode):
        ops = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops.append(str(func))
            return func(*args, **(kwargs or {}))
    with Seen():
        out = mod(x)
    assert _same(out, first) and any("empty" in op for op in Seen.ops)


@pytest.mark.parametrize("M,N,K", [(16, 200, 256), (1, 64, 4096), (8, 64 * 260, 256), (16, 512, 256), (40, 512, 256)])
@pytest.mark.parametrize("bits", [4, 8])
def test_fused_dequantize_allocates_what_it_uses(M, N, K, bits):
    """The result, and for a call in two launches the int32 product: no result that is thrown away because the call turns
    out to need the product's memory."""
    import quik
    from quik_amd import _lib as L
    if isinstance(L.front(), L._NoFront):
        pytest.skip("no native front end")
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    kbytes = K // 2 if bits == 4 else K
    a, b = (torch.randint(-8, 8, (n, kbytes), generator=g, device=DEV, dtype=torch.int8) for n in (M, N))
    if bits == 4:
        a, b = a.view(torch.uint8), b.view(torch.uint8)
    s_row, s_col = ((torch.rand(*s, generator=g, device=DEV) * 0.1).half() for s in ((M, 1), (1, N)))
    y = torch.randn(M, N, generator=g, device=DEV).half()
    op = quik.symmetric.int4FusedDequantize if bits == 4 else quik.symmetric.int8FusedDequantize
    op(a, b, s_row, s_col, y)
    made = torch.cuda.memory_stats()["allocation.all.allocated"]
    got = op(a, b, s_row, s_col, y)
    made = torch.cuda.memory_stats()["allocation.all.allocated"] - made
    need = L.load().quik_fused_dequantize_acc_bytes(M, N, K, bits)
    assert need in (0, M * N * 4) and (need == 0 or M <= 32)
    assert made == (2 if need else 1)
    mm = quik.matmul.int4Matmul if bits == 4 else quik.matmul.int8Matmul
    want = quik.symmetric.dequantize(mm(a, b), s_row, s_col, y, 32)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
