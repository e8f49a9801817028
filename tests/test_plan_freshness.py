"""Plans for the native front end hold only what the module's buffers are when the plan is made.

A layer keeps one descriptor per path (row-major, tile-ordered), and a forward brings only its own up to date.  Here the
library, the packing kernels and the front end are stand-ins on CPU tensors, so that the descriptors a plan receives can
be compared with the module's buffers: addresses, and the contents that the tile-ordered operand was packed from.
"""
import copy
import ctypes
import itertools
import pickle

import pytest
import torch

from quik_amd import _lib as L
from quik_amd import asymmetric, matmul, qlinear
from quik_amd.qlinear import MixedQLinear, SharedQuantizedInput

N, N_IN, F = 24, 160, 32
DECODE, PREFILL = 1, 64     # row-major and tile-ordered path


class Binding:
    def __init__(self):
        self.calls, self.packed, self.plans, self.groups, self.packs = [], {}, [], 0, 0

    # the library
    def quik_layer_workspace_bytes(self, desc, rows):
        return 16

    def quik_layer_forward(self, desc, x, rows, *rest):
        self.calls.append((rows, L.QuikLayer.from_buffer_copy(desc._obj)))
        return 0

    # the packing kernels: an operand that is a copy of what it was made from
    def pack(self, int_weight, fp_weight, colmap, *rest):
        w6 = torch.cat([int_weight.reshape(-1), fp_weight.contiguous().view(torch.uint8).reshape(-1), colmap])
        self.packed[w6.data_ptr()] = w6.clone()
        self.packs += 1
        return w6

    # the front end
    def group(self, shared, fused, plan, methods, members):
        self.groups += 1
        return object()

    def plan(self, module, names, row, tiled, tiled_from, device, bf16, dev, splitk, keep):
        self.plans.append([None if b is None else L.QuikLayer.from_buffer_copy(b) for b in (row, tiled)])
        return object()


def colmap_of(int_indices, fp_indices, cols):
    return torch.cat([int_indices, fp_indices]).to(torch.uint8)


@pytest.fixture
def binding(monkeypatch):
    b = Binding()
    monkeypatch.setattr(L, "load", lambda: b)
    monkeypatch.setattr(L, "_lib", b)
    monkeypatch.setattr(L, "front", lambda: b)
    monkeypatch.setattr(L, "stream", lambda: 0)
    monkeypatch.setattr(qlinear, "_front", None)
    monkeypatch.setattr(asymmetric, "build_colmap", colmap_of)
    monkeypatch.setattr(asymmetric, "colmap_streams", lambda *a: True)
    monkeypatch.setattr(matmul, "_splitk_workspace", lambda *a: (None, 0))
    for name in ("pack_weight_layer", "pack_weight_fp6"):
        monkeypatch.setattr(matmul, name, b.pack)
    return b


def layer(seed, shared=None):
    g = torch.Generator().manual_seed(seed)
    m = MixedQLinear(N_IN, N, shared, fp_features_num=F)
    perm = torch.randperm(N_IN, generator=g)
    m.int_indices.copy_(perm[F:].sort()[0])
    m.fp_indices.copy_(perm[:F])
    m.int_weight.random_(0, 256, generator=g)
    for name in ("weights_scales", "fp_weight", "reduced_w", "bias"):
        getattr(m, name).normal_(generator=g)
    return m


def call(m, rows):
    assert m._forward_one_call(torch.zeros(rows, N_IN, dtype=torch.float16)) is not None


def check(b, m, desc, tiled):
    """`desc` describes the module as it is now."""
    for field in ("int_weight", "weights_scales", "reduced_w", "fp_weight", "bias"):
        t = getattr(m, field)
        assert getattr(desc, field) == (None if t is None else t.data_ptr()), field
    assert desc.colmap == m._column_map().data_ptr()
    colmap = colmap_of(m.int_indices, m.fp_indices, N_IN)
    held = (ctypes.c_uint8 * len(colmap)).from_address(desc.colmap)
    assert bytes(held) == bytes(colmap.tolist())
    if tiled:
        assert torch.equal(b.packed[desc.tiled_weight], b.pack(m.int_weight, m.fp_weight, colmap))


def in_place(m):
    m.load_state_dict(layer(1).state_dict())


def replaced(m):
    m.load_state_dict(layer(1).state_dict(), assign=True)


def one_replaced(m):
    m.bias = layer(1).bias


def no_bias(m):
    m.bias = None


def new_outliers(m):
    other = layer(2)
    m.int_indices.copy_(other.int_indices)
    m.fp_indices.copy_(other.fp_indices)


@pytest.mark.parametrize("change", [in_place, replaced, one_replaced, no_bias, new_outliers])
@pytest.mark.parametrize("before", [(), (DECODE,), (PREFILL,), (DECODE, PREFILL), (PREFILL, DECODE)])
def test_a_plan_holds_current_descriptors(binding, before, change):
    for after in itertools.product((DECODE, PREFILL), repeat=3):
        m = layer(0)
        for rows in before:
            call(m, rows)
        change(m)
        for rows in after:
            call(m, rows)
            check(binding, m, binding.calls[-1][1], rows >= 33)
            row, tiled = binding.plans[-1]
            assert (tiled if rows >= 33 else row) is not None
            for desc, t in ((row, False), (tiled, True)):
                if desc is not None:
                    check(binding, m, desc, t)


@pytest.mark.parametrize("on_class", [False, True])
@pytest.mark.parametrize("first", [DECODE, PREFILL])
def test_no_tiled_copy_stays_with_the_transient_policy(binding, monkeypatch, first, on_class):
    m = layer(0)
    call(m, PREFILL)
    call(m, DECODE)
    assert m.weight_bytes()["tiled"] > 0
    if on_class:
        monkeypatch.setattr(MixedQLinear, "transient_tiled_copy", True)
    else:
        m.transient_tiled_copy = True
    for rows in (first, DECODE, PREFILL, DECODE):
        made = len(binding.plans)
        call(m, rows)
        check(binding, m, binding.calls[-1][1], rows >= 33)
        assert m.weight_bytes()["tiled"] == 0 and True not in m._descs
        if rows >= 33:                                    # each such call packs its own operand: no plan serves it
            assert len(binding.plans) == made and "fast" not in m._descs
        else:
            assert binding.plans[-1][1] is None


MEMBER_BUFFERS = ("int_weight", "weights_scales", "fp_weight", "reduced_w", "bias")


def round_of(b, shared, mods, rows):
    """One round of the group's members; the fused layer it ran through, or None."""
    for m in mods:
        out = shared.group_forward(m, torch.zeros(rows, N_IN, dtype=torch.float16))
        if out is None:
            return None
        assert out.shape == (rows, m.out_features)
    fused = shared._fused
    for name in MEMBER_BUFFERS:
        ts = [getattr(m, name) for m in mods]
        if ts[0] is not None:
            assert torch.equal(getattr(fused, name), torch.cat(ts, dim=1 if name == "reduced_w" else 0)), name
    check(b, fused, b.calls[-1][1], rows >= 33)
    for desc, t in zip(b.plans[-1], (False, True)):
        if desc is not None:
            check(b, fused, desc, t)
    return fused


@pytest.mark.parametrize("how", ["written", "assigned", "loaded"])
@pytest.mark.parametrize("name", MEMBER_BUFFERS + ("fp_indices",))
def test_a_group_sees_every_buffer_of_its_members(binding, monkeypatch, name, how):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    for orders in itertools.product((DECODE, PREFILL), repeat=3):
        shared = SharedQuantizedInput(2)
        mods = [layer(0, shared), layer(0, shared)]
        for rows in orders[:2]:
            assert round_of(binding, shared, mods, rows) is not None
        for m, seed in ((mods[1], 1), (mods[0], 2)):       # one member, then the other
            new = getattr(layer(seed), name).clone()
            if how == "written":
                getattr(m, name).copy_(new)
            elif how == "assigned":
                setattr(m, name, new)
            else:
                m.load_state_dict({name: new}, assign=True, strict=False)
            for rows in orders[1:]:
                fused = round_of(binding, shared, mods, rows)
                # (members with other outlier columns have no quantized input in common)
                assert (fused is None) == (name == "fp_indices"), (name, how)


@pytest.mark.parametrize("switch", [("fused", False), ("fuse_shared_groups", False), ("sym_divisor", 7.0), ("six_bit_path", False),
                                    ("transient_tiled_copy", True)])
def test_a_group_sees_the_switches_of_its_members(binding, monkeypatch, switch):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    name, value = switch
    shared = SharedQuantizedInput(2)
    mods = [layer(0, shared), layer(0, shared)]
    for rows in (DECODE, PREFILL):
        round_of(binding, shared, mods, rows)
    assert all("fast" in m._descs for m in mods)
    for k, m in enumerate(mods):
        setattr(m, name, value)
        made = binding.groups
        fused = round_of(binding, shared, mods, DECODE)
        if name == "fuse_shared_groups":                  # the member's own forward asks for this one
            assert binding.groups == made and "fast" not in m._descs and shared._fast is None
        elif name == "fused" or (k == 0 and name in ("sym_divisor", "six_bit_path")):
            assert fused is None                          # the members differ, or one replays the op sequence
        elif name != "transient_tiled_copy" or k == 0:
            assert getattr(fused, name) == value
    if name == "transient_tiled_copy":
        assert round_of(binding, shared, mods, PREFILL).weight_bytes()["tiled"] == 0


class Memory:
    """Tensors over one piece of memory, as an allocator hands a freed block out again: same address, same version."""

    def __init__(self, like):
        self.bytes, self.like = bytearray(like.numel() * like.element_size()), (like.dtype, like.shape)

    def tensor(self, values):
        self.bytes[:] = values.contiguous().view(torch.uint8).numpy().tobytes()
        return torch.frombuffer(self.bytes, dtype=self.like[0]).view(self.like[1])


def set_attribute(m, name, memory, values):
    setattr(m, name, None)
    setattr(m, name, memory.tensor(values))


def set_buffer(m, name, memory, values):          # (as Module.to and load hooks do)
    m._buffers[name] = None
    m._buffers[name] = memory.tensor(values)


def set_data(m, name, memory, values):
    getattr(m, name).data = torch.empty(0, dtype=values.dtype)
    getattr(m, name).data = memory.tensor(values)


@pytest.mark.parametrize("setter", [set_attribute, set_buffer, set_data])
@pytest.mark.parametrize("name", MEMBER_BUFFERS + ("int_indices",))
def test_a_buffer_that_got_the_address_of_a_freed_one(binding, name, setter):
    m = layer(0)
    memory = Memory(getattr(m, name))
    setter(m, name, memory, getattr(m, name).clone())
    for rows in (PREFILL, DECODE, PREFILL):
        call(m, rows)
    where = getattr(m, name).data_ptr()
    setter(m, name, memory, getattr(layer(2), name))
    assert getattr(m, name).data_ptr() == where
    for rows in (DECODE, PREFILL, PREFILL):
        call(m, rows)
        check(binding, m, binding.calls[-1][1], rows >= 33)
        for desc, t in zip(binding.plans[-1], (False, True)):
            assert desc is None or check(binding, m, desc, t) is None


def test_stamps_do_not_travel(binding):
    m = layer(0)
    call(m, PREFILL)
    for other in (copy.deepcopy(m), pickle.loads(pickle.dumps(m))):
        packs = binding.packs
        call(other, PREFILL)
        assert binding.packs > packs
        check(binding, other, binding.calls[-1][1], True)


def test_forwards_under_inference_mode(binding):
    m = layer(0)
    with torch.inference_mode():       # (what a forward makes for itself has no version there)
        for rows in (PREFILL, DECODE, PREFILL):
            call(m, rows)
    packs = binding.packs
    call(m, PREFILL)
    assert binding.packs == packs
    check(binding, m, binding.calls[-1][1], True)


@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
@pytest.mark.parametrize("method", ["_forward_one_call", "_six_bit_ok", "_descriptor", "_weight6", "_column_map"])
def test_an_override_is_called_by_every_forward(binding, monkeypatch, method, where):
    real, seen = getattr(MixedQLinear, method), []

    def override(self, *args):
        seen.append(method)
        return real(self, *args)

    m = layer(0)
    for rows in (PREFILL, DECODE):
        call(m, rows)
    if where == "subclass":
        m.__class__ = type("Sub", (MixedQLinear,), {method: override})
    elif where == "class":
        monkeypatch.setattr(MixedQLinear, method, override)
    else:
        setattr(m, method, override.__get__(m))
    for rows in (PREFILL, DECODE, PREFILL):
        del seen[:]
        call(m, rows)
        assert "fast" not in m._descs
        assert seen or method in ("_weight6", "_column_map")    # (what a descriptor is made from once)


@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
@pytest.mark.parametrize("method", ["group_forward", "_fused_layer"])
def test_an_override_of_the_group_is_called_by_every_round(binding, monkeypatch, method, where):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    real = getattr(SharedQuantizedInput, method)

    def override(self, *args):
        return real(self, *args)

    shared = SharedQuantizedInput(2)
    mods = [layer(0, shared), layer(0, shared)]
    round_of(binding, shared, mods, DECODE)
    if where == "subclass":
        shared.__class__ = type("Sub", (SharedQuantizedInput,), {method: override})
    elif where == "class":
        monkeypatch.setattr(SharedQuantizedInput, method, override)
    else:
        setattr(shared, method, override.__get__(shared))
    made = binding.groups
    round_of(binding, shared, mods, DECODE)
    assert binding.groups == made and shared._fast is None
