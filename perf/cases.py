"""The calls that programs make of this library, as cases that can be timed and checked.

A case is one call of a public entry point on tensors that lie in HBM: the decode, batched-decode, prefill, quantised
and batched matrix products that a transformer's layers are made of, and the reference's own matmul shapes. ``listed``
has one of each kind; ``draw`` gives others of the same kinds, over the range of sizes that each kind has in use.
Sizes follow the benchmark's configurations (C1 to C5), its dispatch sweep, the reference's perf shapes and generic
transformer widths.
"""
import math

import torch

import kudnn_amd as K
import kudnn_amd.torch_linear as kl

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "s8": torch.int8, "u8": torch.uint8,
          "s32": torch.int32}
_DT = {"f32": K.F32, "bf16": K.BF16, "f16": K.F16, "s8": K.S8, "u8": K.U8, "s32": K.S32}
_ACT = {"none": K.ACT_UNIMPLEMENTED, "relu": K.ACT_RELU, "swish": K.ACT_SWISH, "gelu_tanh": K.ACT_GELU_TANH}
_BIN = {"none": K.BIN_NONE, "add": K.BIN_ADD, "mul": K.BIN_MUL}


def _case(op, m, k, n, dtype, wdtype=None, ydtype=None, batch=1, layout="BA", bias=False, act="none", binary="none",
          alpha=1.0):
    return {"op": op, "m": m, "k": k, "n": n, "batch": batch, "dtype": dtype, "wdtype": wdtype or dtype,
            "ydtype": ydtype or dtype, "layout": layout, "bias": bias, "act": act, "binary": binary, "alpha": alpha}


def _named(name, **kw):
    return dict(_case(**kw), name=name)


def listed():
    return [
        # One token through a projection of a PyTorch model: the smallest call, in which the launch and the host count.
        _named("token_torch", op="torch", m=1, k=4096, n=4096, dtype="bf16", binary="mul"),
        # Sixteen sequences decoded together through the gate of an MLP (C4's largest shape): the weight is streamed.
        _named("decode_m16", op="postops", m=16, k=4096, n=14336, dtype="bf16", binary="mul"),
        # Four sequences against a weight kept in 8 bits (W8A16), which halves what decode has to stream.
        _named("decode_w8a16", op="gemm", m=4, k=4096, n=4096, dtype="f16", wdtype="s8", bias=True, alpha=2.0 ** -7),
        # A serving batch between decode and prefill: 64 rows up the MLP, GELU fused.
        _named("batch_64", op="postops", m=64, k=4096, n=11008, dtype="bf16", act="gelu_tanh"),
        # A prompt chunk of a length that is no multiple of anything, down the MLP, with both outputs of LinearResFWD.
        _named("chunk_500_res", op="res", m=500, k=11008, n=4096, dtype="bf16", bias=True, binary="add"),
        # Prefill up the MLP: Linear + GELU(tanh) + residual, the benchmark's headline (C3).
        _named("prefill_c3", op="postops", m=4096, k=4096, n=11008, dtype="bf16", act="gelu_tanh", binary="add"),
        # A batch of long prompts with the weight stored [K][N] and a 3-D source, bias and SiLU (C5): the largest call.
        _named("prefill_c5", op="act", m=2048, k=5120, n=13824, batch=8, dtype="bf16", layout="AB", bias=True,
               act="swish"),
        # A small fp32 layer, bound by latency (C1).
        _named("f32_c1", op="act", m=128, k=1024, n=1024, dtype="f32", bias=True, act="relu"),
        # A large fp32 layer with SiLU (C2).
        _named("f32_c2", op="act", m=2048, k=4096, n=4096, dtype="f32", bias=True, act="swish"),
        # The reference's matmul test on one of its perf shapes, whose K is no multiple of a tile; weight [K][N].
        _named("matmul_ragged", op="gemm", m=4096, k=3256, n=1152, dtype="bf16", layout="AB", bias=True),
        # A quantised layer: u8 activations and s8 weights into s32 (W8A8).
        _named("w8a8", op="gemm", m=1024, k=4096, n=4096, dtype="u8", wdtype="s8", ydtype="s32", bias=True),
        # A product per attention head: 32 heads, 128 wide, 1024 x 1024 scores.
        _named("heads_qk", op="gemm", m=1024, k=128, n=1024, batch=32, dtype="bf16", alpha=2.0 ** -3),
    ]


def _size(rng, lo, hi, steps=(128, 128, 128, 64, 64, 8, 8, 1)):
    """A size of [lo, hi], spread over its logarithm, usually a multiple of a tile's side and at times odd."""
    step = rng.choice(steps)
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _drawn(rng):
    kind = rng.choice(["torch", "decode", "decode", "w8a16", "batch", "batch", "chunk", "chunk", "prefill", "prefill",
                       "f32_small", "f32", "matmul", "w8a8", "heads"])
    k, n = _size(rng, 2048, 14336), _size(rng, 2048, 14336)
    bias, act = rng.random() < 0.5, rng.choice(["none", "relu", "swish", "gelu_tanh"])
    layout, half = rng.choice(["BA", "BA", "AB"]), rng.choice(["bf16", "bf16", "f16"])
    if kind == "torch":
        return _case("torch", rng.randint(1, 16), k, n, rng.choice(["bf16", "bf16", "f32"]), bias=bias, act=act,
                     binary=rng.choice(["none", "add", "mul"]))
    if kind == "decode":
        return _case("postops", rng.randint(1, 16), k, _size(rng, 2048, 28672), half, bias=bias, act=act,
                     binary=rng.choice(["none", "add", "mul"]))
    if kind == "w8a16":
        return _case("gemm", _size(rng, 1, 256, (1,)), k, n, "f16", rng.choice(["s8", "s8", "u8"]), bias=bias,
                     alpha=2.0 ** -7)
    if kind == "batch":
        return _case("postops", _size(rng, 17, 256, (1, 8, 16)), k, n, half, layout=layout, bias=bias, act=act,
                     binary=rng.choice(["none", "add", "mul"]))
    if kind == "chunk":
        m = _size(rng, 257, 2048, (1, 8, 64))
        if rng.random() < 0.5:
            return _case("res", m, k, n, half, layout=layout, bias=bias, binary="add")
        return _case("act", m, k, n, half, layout=layout, bias=bias, act=act if act != "none" else "swish")
    if kind == "prefill":
        return _case("postops", _size(rng, 2048, 8192, (1, 64, 256)), _size(rng, 2048, 8192), _size(rng, 2048, 16384),
                     half, layout=layout, bias=bias, act=act, binary=rng.choice(["none", "add", "mul"]))
    if kind == "f32_small":
        return _case("act", _size(rng, 16, 512, (1, 8, 16)), _size(rng, 256, 4096), _size(rng, 256, 4096), "f32",
                     layout=layout, bias=True, act=rng.choice(["relu", "swish", "gelu_tanh"]))
    if kind == "f32":
        return _case("act", _size(rng, 512, 4096, (1, 64, 128)), _size(rng, 1024, 5120), _size(rng, 1024, 5120), "f32",
                     layout=layout, bias=bias, act=rng.choice(["relu", "swish", "gelu_tanh"]))
    if kind == "matmul":
        return _case("gemm", _size(rng, 1024, 4096), _size(rng, 512, 5120, (8, 8, 1)), _size(rng, 512, 8192), half,
                     layout="AB", bias=True)
    if kind == "w8a8":
        return _case("gemm", _size(rng, 16, 4096, (1, 16, 64)), k, n, rng.choice(["u8", "s8"]), "s8", "s32", bias=bias)
    return _case("gemm", _size(rng, 128, 2048, (1, 64, 128)), rng.choice([64, 80, 96, 128]), _size(rng, 128, 2048),
                 half, batch=rng.randint(8, 64), layout=rng.choice(["BA", "AB"]), alpha=2.0 ** -3)


_MOST_FLOPS = 2.0 * 16384 * 5120 * 13824
_MOST_F32_FLOPS = 1.5e11


def draw(rng):
    while True:
        case = _drawn(rng)
        if work(case)["flops"] <= (_MOST_F32_FLOPS if case["dtype"] == "f32" else _MOST_FLOPS):
            return case


def _normal(gen, shape, std, dtype):
    return (torch.randn(*shape, device="cuda", generator=gen) * std).to(_TORCH[dtype])


def _weight_batched(case):
    # a product per head has a right operand per batch; a layer's weight is shared
    return case["op"] == "gemm" and case["batch"] > 1


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    xs = (b, m, k) if b > 1 else (m, k)
    ws = (n, k) if case["layout"] == "BA" else (k, n)
    ws = (b,) + ws if _weight_batched(case) else ws
    t = {}
    if case["dtype"] in ("s8", "u8"):
        # quantised activations: bell-shaped around the zero point
        z = 128.0 if case["dtype"] == "u8" else 0.0
        t["x"] = (torch.randn(*xs, device="cuda", generator=gen) * 32.0 + z).round_().clamp_(z - 127, z + 127).to(
            _TORCH[case["dtype"]])
    else:
        t["x"] = _normal(gen, xs, 1.0, case["dtype"])
    if case["wdtype"] in ("s8", "u8"):
        z = 128.0 if case["wdtype"] == "u8" else 0.0
        t["w"] = (torch.randn(*ws, device="cuda", generator=gen) * 32.0 + z).round_().clamp_(z - 127, z + 127).to(
            _TORCH[case["wdtype"]])
    else:
        t["w"] = _normal(gen, ws, 1.0 if _weight_batched(case) else 0.02, case["wdtype"])
    if case["bias"]:
        if case["ydtype"] == "s32":
            t["bias"] = torch.randint(-65536, 65536, (n,), device="cuda", generator=gen, dtype=torch.int32)
        else:
            t["bias"] = _normal(gen, (n,), 0.1, _bias_dtype(case))
    if case["binary"] != "none":
        t["src"] = _normal(gen, xs[:-1] + (n,), 1.0, case["ydtype"])
    return t


def _bias_dtype(case):
    # KuDNN::Gemm takes the bias of a 16-bit product in f32; the fused layers are given the layer's own type
    return "f32" if case["op"] == "gemm" and case["ydtype"] != "s32" else case["ydtype"]


def prepare(case, seed):
    s = _inputs(case, seed)
    s["op"], s["alpha"] = case["op"], case["alpha"]
    b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    if case["op"] == "torch":
        layer = kl.KudnnLinear(k, n, case["bias"], None if case["act"] == "none" else case["act"], None,
                               None if case["binary"] == "none" else case["binary"], device="cuda",
                               dtype=_TORCH[case["dtype"]])
        with torch.no_grad():
            layer.weight.copy_(s.pop("w"))
            if case["bias"]:
                layer.bias.copy_(s.pop("bias"))
        s["layer"] = layer
        return s
    lead = [b] if b > 1 else []
    wlead = ([b] if _weight_batched(case) else [1]) if b > 1 else []
    wlayout = {("BA", 0): "BA", ("BA", 1): "ACB", ("AB", 0): "AB", ("AB", 1): "ABC"}[(case["layout"], len(lead))]
    dx = K.desc(lead + [m, k], _DT[case["dtype"]])
    dw = K.desc(wlead + [k, n], _DT[case["wdtype"]], wlayout)
    dy = K.desc(lead + [m, n], _DT[case["ydtype"]])
    db = K.desc([1] * (len(lead) + 1) + [n], _DT[_bias_dtype(case)]) if case["bias"] else None
    s["y"] = torch.empty(lead + [m, n], device="cuda", dtype=_TORCH[case["ydtype"]])
    if case["op"] == "gemm":
        s["plan"] = K.Gemm(dx, dw, dy, db)
    elif case["op"] == "act":
        s["plan"] = K.LinearActivation(dx, dw, dy, db, alpha=1.0 if case["act"] == "swish" else 0.0,
                                       kind=_ACT[case["act"]])
    elif case["op"] == "res":
        s["plan"] = K.LinearRes(dx, dw, dy, db, dy, dy, kind=K.RES_IDENTIAL)
        s["sum"] = torch.empty_like(s["y"])
    else:
        s["plan"] = K.LinearPostOps(dx, dw, dy, db, act=_ACT[case["act"]],
                                    act_alpha=1.0 if case["act"] == "swish" else 0.0, binary=_BIN[case["binary"]],
                                    src=dy if case["binary"] != "none" else None)
    return s


def run(state):
    op, x, y = state["op"], state["x"], state.get("y")
    if op == "torch":
        with torch.inference_mode():
            return state["layer"](x, state.get("src"))
    if op == "gemm":
        state["plan"].run(x, state["w"], y, state.get("bias"), alpha=state["alpha"])
    elif op == "act":
        state["plan"].run(x, state["w"], y, state.get("bias"))
    elif op == "res":
        state["plan"].run(x, state["w"], y, state.get("bias"), state["src"], state["sum"])
        return y, state["sum"]
    else:
        state["plan"].run(x, state["w"], y, state.get("bias"), state.get("src"))
    return y


_BYTES = {"f32": 4, "s32": 4, "bf16": 2, "f16": 2, "s8": 1, "u8": 1}


def work(case):
    b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    out = b * m * n * _BYTES[case["ydtype"]]
    total = b * m * k * _BYTES[case["dtype"]] + out
    total += (b if _weight_batched(case) else 1) * k * n * _BYTES[case["wdtype"]]
    total += n * _BYTES[_bias_dtype(case)] if case["bias"] else 0
    total += out if case["binary"] != "none" else 0
    total += out if case["op"] == "res" else 0
    return {"bytes": total, "flops": 2 * b * m * k * n}


def tolerance(case):
    if case["ydtype"] == "s32":
        return "exact"
    # Another order of the f32 sums moves an output by its own rounding to the output type, and in bf16 by one more
    # where a fused stage rounds before the last.
    if case["ydtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["ydtype"] == "f16":
        return {"rel": 2e-3, "max": 1e-2}
    return {"rel": 1e-2, "max": 5e-2}


def exact(case, seed):
    t = _inputs(case, seed)
    x, w = t["x"].double(), t["w"].double()
    if case["layout"] == "BA":
        w = w.transpose(-1, -2).contiguous()
    y = torch.matmul(x, w) * case["alpha"]
    del x, w
    if case["bias"]:
        y += t["bias"].double()
    if case["ydtype"] == "s32":
        return y.round_().to(torch.int32)  # every term and partial sum is an integer far below 2^53
    if case["act"] == "relu":
        y = torch.relu_(y)
    elif case["act"] == "swish":
        y = y * torch.sigmoid(y)
    elif case["act"] == "gelu_tanh":
        y = torch.nn.functional.gelu(y, approximate="tanh")
    if case["op"] == "res":
        return y, y + t["src"].double()
    if case["binary"] == "add":
        y = y + t["src"].double()
    elif case["binary"] == "mul":
        y = y * t["src"].double()
    return y
