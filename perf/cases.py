"""The calls whose speed matters to a program that uses this package, with their inputs.

`listed()` names them, `draw(rng)` gives further calls of the same ranges, `prepare` makes what a program holds before
the call (layers built with `from_float`, activations), `run` is the call.  Activations are N(0, 1) with the outlier
columns scaled by 50, weight codes uniform over their range, column scales U(0.001, 0.01), outlier weights N(0, 0.02).

Kinds of call:
  layer   MixedQLinear.forward, the layer a quantized model consists of
  group   the members of one SharedQuantizedInput (q/k/v, gate/up), called one after the other on one input
  ops     the stand-alone operations in the order the layer is made of: asymmetric.quantize, the outlier product,
          the integer product, asymmetric.dequantize
  fused   asymmetric.int4FusedDequantize / int8FusedDequantize on quantized operands
"""
import torch

import quik
from quik_amd.qlinear import MixedQLinear, SharedQuantizedInput

# layer shapes in -> out of the 7B, 13B and 70B configurations of this repository
SHAPES4 = ((4096, 4096), (4096, 11008), (5120, 5120), (5120, 13824), (8192, 8192), (8192, 1024), (8192, 28672))
SHAPES8 = ((11008, 4096), (13824, 5120), (28672, 8192))


def _case(kind, rows, n_in, out, fp=256, bits=4, symm=False, dtype="float16", bias=False, members=1, out2=0):
    """`members` layers in a group: the first has `out` columns, the others `out2`."""
    return {"kind": kind, "rows": rows, "in": n_in, "out": out, "fp": fp, "bits": bits, "symm": symm, "dtype": dtype,
            "bias": bias, "members": members, "out2": out2}


def listed():
    return [
        # one sequence, token by token: the smallest projection and the largest
        dict(_case("layer", 1, 4096, 4096), name="decode_1_q"),
        dict(_case("layer", 1, 8192, 28672), name="decode_1_gate"),
        # a few sequences decoded together, the 8-bit projection
        dict(_case("layer", 16, 13824, 5120, bits=8), name="decode_16_down8"),
        # the decode step of a 64-sequence batch: q, k and v of a grouped-query layer from one quantized input
        dict(_case("group", 64, 8192, 8192, members=3, out2=1024), name="decode_64_qkv"),
        # a short prompt
        dict(_case("layer", 128, 5120, 13824), name="prompt_128_gate"),
        # the operations by themselves, as a program with a layer class of its own calls them
        dict(_case("ops", 512, 4096, 4096, fp=128), name="ops_512"),
        # quantized operands straight to 16-bit outputs
        dict(_case("fused", 256, 4096, 4096, fp=0), name="fused_op_256"),
        # a prompt of no particular length, a width that is no multiple of the tiles, a bias
        dict(_case("layer", 300, 4544, 4544, fp=128, bias=True), name="prompt_300_odd_width"),
        # bfloat16 activations, gate and up together
        dict(_case("group", 777, 4096, 11008, dtype="bfloat16", members=2, out2=11008), name="prompt_777_gate_up_bf16"),
        # prefill: a narrow key projection with symmetric activations, the wide projection, the 8-bit one over a batch
        dict(_case("layer", 2048, 8192, 1024, symm=True), name="prefill_2048_k_symm"),
        dict(_case("layer", 2048, 8192, 28672), name="prefill_2048_gate"),
        dict(_case("layer", 8192, 28672, 8192, bits=8), name="prefill_8192_down8"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("layer",) * 6 + ("group", "group", "ops", "fused"))
    bits = rng.choice((4, 4, 8))
    rows = _log(rng, 1, 8192 if kind == "layer" else 2048)
    if rng.random() < 0.6:
        n_in, out = rng.choice(SHAPES4 + SHAPES8[:2] if bits == 4 else SHAPES8)
    else:
        n_in, out = 64 * _log(rng, 16, 224), 8 * _log(rng, 64, 2048)
    fp = rng.choice((0, 64, 128, 256, 256, 256, 32 * rng.randint(1, 16)))
    symm = bits == 4 and kind in ("layer", "group") and rng.random() < 0.2
    dtype = "bfloat16" if kind in ("layer", "group") and not symm and rng.random() < 0.2 else "float16"
    bias = kind in ("layer", "group") and rng.random() < 0.25
    members = rng.choice((2, 3)) if kind == "group" else 1
    out2 = 0 if members == 1 else out if members == 2 else max(256, out // 8 // 8 * 8)
    if kind == "fused":
        fp = 0
    while rows * n_in * (out + (members - 1) * out2) > 8192 * 28672 * 8192:
        rows = max(1, rows // 2)
    return _case(kind, rows, n_in, out, fp, bits, symm, dtype, bias, members, out2)


def _weights(case, out, fp_idx, int_idx, g):
    """Fake-quantized weight matrix [out, in] and its column scales, as a calibration leaves them."""
    dt, dev = getattr(torch, case["dtype"]), "cuda"
    scales = (torch.rand(out, 1, generator=g, device=dev) * 0.009 + 0.001).to(dt)
    lo, hi = (-8, 8) if case["bits"] == 4 else (-127, 128)
    w = torch.randint(lo, hi, (out, case["in"]), generator=g, device=dev, dtype=torch.int16).to(dt)
    w *= scales
    if case["fp"]:
        w[:, fp_idx] = 0.02 * torch.randn(out, case["fp"], generator=g, device=dev).to(dt)
    return w, scales


def _layer(case, out, fp_idx, int_idx, g, shared):
    w, scales = _weights(case, out, fp_idx, int_idx, g)
    lin = torch.nn.Linear(case["in"], out, bias=False, device="meta")
    if case["bias"]:
        lin.bias = torch.nn.Parameter(torch.randn(out, generator=g, device="cuda").to(w.dtype), requires_grad=False)
    return MixedQLinear.from_float(lin, w, scales, shared, fp_idx, symm=case["symm"], bits=case["bits"]).to("cuda")


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = getattr(torch, case["dtype"])
    rows, n_in, out, bits = case["rows"], case["in"], case["out"], case["bits"]
    if case["kind"] == "fused":
        lo, hi = (0, 256) if bits == 4 else (-128, 128)
        code_t, kb = (torch.uint8, n_in // 2) if bits == 4 else (torch.int8, n_in)
        a = torch.randint(lo, hi, (rows, kb), generator=g, device="cuda", dtype=torch.int16).to(code_t)
        b = torch.randint(lo, hi, (out, kb), generator=g, device="cuda", dtype=torch.int16).to(code_t)

        def half(*shape):
            return torch.rand(*shape, generator=g, device="cuda").half()
        # (8-bit sums reach beyond what a half holds: column scales are small, sums of a trained layer are too)
        if bits == 8:
            a >>= 3
            b >>= 3
        return {"kind": "fused", "bits": bits, "args": (a, b, half(rows, 1) * 0.1, half(1, out) * 0.01, 8.0 if bits == 4
                else 128.0, -half(rows, 1), half(1, out), half(rows, out))}
    fp_idx = torch.randperm(n_in, generator=g, device="cuda")[:case["fp"]]
    keep = torch.ones(n_in, dtype=torch.bool, device="cuda")
    keep[fp_idx] = False
    int_idx = torch.arange(n_in, device="cuda")[keep]
    x = torch.randn(rows, n_in, generator=g, device="cuda")
    x[:, fp_idx] *= 50
    x = x.to(dt)
    if case["kind"] == "ops":
        layer = _layer(case, out, fp_idx, int_idx, g, None)
        return {"kind": "ops", "bits": bits, "x": x, "int_idx": int_idx, "fp_idx": fp_idx, "w": layer.int_weight,
                "scales": layer.weights_scales, "reduced_w": layer.reduced_w,
                "fp_w": layer.fp_weight if case["fp"] else None,
                "zeros": None if case["fp"] else torch.zeros(rows, out, dtype=dt, device="cuda")}
    shared = SharedQuantizedInput(case["members"])
    outs = [out] + [case["out2"]] * (case["members"] - 1)
    return {"kind": case["kind"], "x": x, "layers": [_layer(case, n, fp_idx, int_idx, g, shared) for n in outs]}


def run(state):
    kind = state["kind"]
    if kind == "fused":
        op = quik.asymmetric.int4FusedDequantize if state["bits"] == 4 else quik.asymmetric.int8FusedDequantize
        return op(*state["args"])
    if kind == "ops":
        q, meta, fp_x = quik.asymmetric.quantize(state["x"], state["int_idx"], state["fp_idx"], state["bits"])
        y = state["zeros"] if state["fp_w"] is None else torch.nn.functional.linear(fp_x, state["fp_w"])
        acc = (quik.matmul.int4Matmul if state["bits"] == 4 else quik.matmul.int8Matmul)(q, state["w"])
        out = quik.asymmetric.dequantize(acc, meta, state["scales"], state["reduced_w"], y, state["bits"])
        return {"q": q, "meta": meta, "acc": acc, "out": out}
    x = state["x"]
    return [layer(x) for layer in state["layers"]]


def work(case):
    rows, n_in, fp = case["rows"], case["in"], case["fp"]
    out = case["out"] + (case["members"] - 1) * case["out2"]
    k, code = n_in - fp, case["bits"] / 8
    flops = 2 * rows * out * n_in
    weights = out * (k * code + 2 * fp) + 4 * out
    if case["kind"] == "fused":
        return {"bytes": rows * k * code + weights + 4 * rows + 4 * rows * out, "flops": flops}
    moved = 2 * rows * n_in + weights + 2 * rows * out
    if case["kind"] == "ops":  # the codes and the integer sums are results too
        moved += rows * k * code + 4 * rows * out
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # 16-bit results of exact integer sums and 32-bit outlier sums: the rounding of the result, and of the outlier
    # product where an implementation keeps it in 16 bits.  Codes and integer sums are exact.
    if case["dtype"] == "bfloat16":
        return {"rel": 8e-3, "max": 3e-2}
    return {"rel": 1e-3, "max": 1e-2}
