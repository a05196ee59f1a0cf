"""What the speed of this framework is measured on: the quantized-weight work of one model step.

Each case is work that a program running a quantized ONNX model on this library repeats for every
token, prompt or batch, through the C ABI (`transmuter_amd._lib.lib()`, the package's binding of
include/transmuter_hip.h) over weights packed once, into output buffers that the program keeps.
Launch-bound steps (decode) are captured once into a HIP graph and replayed, as a serving loop does;
the others are called directly. Kinds of cases:

  op      one MatMulNBits node.
  layers  the MatMulNBits projections of a decoder's layers: q/k/v merged, attention output,
          gate/up merged, down (what the load-time move and merge leave of a layer).
  vocab   the two large-vocabulary nodes of a step: GatherBlockQuantized of the prompt's ids and
          the lm_head over the last positions.
  qmoe    one QMoE node (routing, expert products, weighted sum).
  int8    a dynamically quantized linear layer: DynamicQuantizeLinear, MatMulInteger over a
          prepared B, DequantizeLinear of the s32 sums.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from transmuter_amd import Context, PackedWeight
from transmuter_amd import _lib
from transmuter_amd._lib import lib
from transmuter_amd.moe import ExpertWeight
from transmuter_amd.packed import Int8Weight

CODE = {"f32": _lib.F32, "f16": _lib.F16, "bf16": _lib.BF16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
DEVICE = "cuda"

_CTX = None


def _ctx() -> Context:
    """The program's one context (device and stream)."""
    global _CTX
    if _CTX is None:
        torch.cuda.init()
        _CTX = Context(0)
    return _CTX


# ---------------------------------------------------------------- the cases


def _layers(name, m, layers, hidden, q, kv, inter, dtype, *, weights=None, bits=4, block=32, zp="packed"):
    # Up to 64 rows a step is decode: bound by launches, so a program replays it as one graph.
    return {"name": name, "kind": "layers", "m": m, "layers": layers, "hidden": hidden, "q": q, "kv": kv,
            "inter": inter, "bits": bits, "block": block, "zp": zp, "dtype": dtype, "weights": weights or dtype,
            "graph": m <= 64}


def listed() -> list[dict]:
    qwen = dict(hidden=1024, q=2048, kv=1024, inter=3072)  # Qwen3-0.6B
    smol = dict(hidden=2048, q=2048, kv=512, inter=11008)  # SmolLM3-3B
    return [
        # The smallest call: one f32 projection of one token, as an f32 export of a small model has it.
        {"name": "op f32 1x1024x3072", "kind": "op", "m": 1, "k": 1024, "n": 3072, "bits": 4, "block": 32,
         "zp": "none", "dtype": "f32", "weights": "f32", "bias": False},
        # One user's chat: every projection of a whole decode step for one token.
        _layers("decode f16 m1", 1, 28, dtype="f16", **qwen),
        # A server decoding for 32 users at once.
        _layers("decode f16 m32", 32, 28, dtype="f16", **qwen),
        # Small decode batches of models exported in bf16 and in f32 (scales in the same type; f32
        # exports quantize symmetrically: no zero points).
        _layers("decode bf16 m8", 8, 28, dtype="bf16", **qwen),
        _layers("decode f32 m16", 16, 28, dtype="f32", zp="none", **qwen),
        # A chat turn's prompt and a long document's chunk through one layer of a 3B model.
        _layers("prefill f16 m256", 256, 1, dtype="f16", **smol),
        _layers("prefill f16 m2048", 2048, 1, dtype="f16", **smol),
        # A prompt of odd length through one layer of a small f32 export.
        _layers("prefill f32 m509", 509, 1, dtype="f32", zp="none", **qwen),
        # A step's two vocabulary nodes: 8 prompts of 512 tokens embedded, 8 last positions scored.
        {"name": "vocab f16 ids4096 m8", "kind": "vocab", "rows": 151936, "dim": 1024, "ids": 4096, "m": 8, "bits": 4,
         "block": 32, "dtype": "f16"},
        # The mixture-of-experts layer of Qwen3-30B-A3B: a prompt's 512 tokens, and a decode batch of 8.
        {"name": "qmoe f16 t512", "kind": "qmoe", "tokens": 512, "experts": 128, "k": 8, "hidden": 2048, "inter": 768,
         "bits": 4, "block": 32, "activation": "swiglu", "dtype": "f16"},
        {"name": "qmoe f16 t8", "kind": "qmoe", "tokens": 8, "experts": 128, "k": 8, "hidden": 2048, "inter": 768,
         "bits": 4, "block": 32, "activation": "swiglu", "dtype": "f16"},
        # A dynamically quantized int8 layer over 2048 rows (an encoder's batch).
        {"name": "int8 2048x2048x2048", "kind": "int8", "m": 2048, "k": 2048, "n": 2048, "b": "s8", "b_zero": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _to(value, multiple):
    return max(multiple, value // multiple * multiple)


def draw(rng) -> dict:
    kind = rng.choice(["op", "op", "layers", "layers", "layers", "vocab", "qmoe", "int8"])
    bits = rng.choice([4, 4, 4, 4, 8, 8, 2])
    block = rng.choice([16, 32, 32, 32, 64, 128])
    dtype = rng.choice(["f16", "f16", "bf16", "f32"])
    if kind == "op":
        # K in steps of 16 (partial blocks and chunks among them), N any size, odd ones too.
        m = _log(rng, 1, 1024)
        k = _to(_log(rng, 256, 8192), 16)
        n = _log(rng, 64, 16384)
        if rng.random() < 0.5:
            n = _to(n, 16)
        weights = dtype if rng.random() < 0.85 else rng.choice(["f16", "f32"])
        return {"kind": "op", "m": m, "k": k, "n": n, "bits": bits, "block": block,
                "zp": rng.choice(["packed", "packed", "none", "float"]), "dtype": dtype, "weights": weights,
                "bias": rng.random() < 0.3}
    if kind == "layers":
        hidden = _to(_log(rng, 384, 4096), 64)
        case = _layers("", _log(rng, 1, 2048), rng.randint(1, 4), hidden, _to(int(hidden * rng.uniform(0.75, 2)), 64),
                       _to(_log(rng, 128, 1024), 64), _to(int(hidden * rng.uniform(2, 4)), 32), dtype,
                       bits=rng.choice([4, 4, 4, 8]), block=rng.choice([32, 32, 64, 128]),
                       zp=rng.choice(["packed", "none"]))
        del case["name"]
        if case["m"] > 256:
            case["layers"] = 1
        return case
    if kind == "vocab":
        dim = _to(_log(rng, 384, 2048), 128)
        return {"kind": "vocab", "rows": _log(rng, 20000, 151936), "dim": dim, "ids": _log(rng, 1, 8192),
                "m": rng.randint(1, 16), "bits": rng.choice([4, 4, 8]), "block": rng.choice([32, 64, 128]),
                "dtype": rng.choice(["f16", "f16", "f32"])}
    if kind == "qmoe":
        experts = rng.choice([8, 16, 32, 64, 128])
        return {"kind": "qmoe", "tokens": _log(rng, 1, 512), "experts": experts, "k": rng.randint(1, min(8, experts)),
                "hidden": _to(_log(rng, 512, 2048), 64), "inter": _to(_log(rng, 256, 1024), 32),
                "bits": rng.choice([4, 4, 8]), "block": rng.choice([32, 64, 128]),
                "activation": rng.choice(["swiglu", "swiglu", "silu", "gelu"]), "dtype": "f16"}
    return {"kind": "int8", "m": _log(rng, 1, 4096), "k": _to(_log(rng, 256, 4096), 16), "n": _log(rng, 64, 4096),
            "b": rng.choice(["s8", "u8"]), "b_zero": rng.random() < 0.5}


# ---------------------------------------------------------------- inputs


def _gen(seed, *path):
    """A generator for one input: every input of a case has its own, made from the seed."""
    x = (int(seed) + 1) * 1000003
    for p in path:
        x = (x * 1000003 + int(p) + 1) % (1 << 62)
    return torch.Generator(device=DEVICE).manual_seed(x)


def _pack_rows(q, bits):
    """u8 values [R, C] packed lowest bits first into rows of ceil(C * bits / 8) bytes."""
    per = 8 // bits
    r, c = q.shape
    q = torch.nn.functional.pad(q, (0, -c % per)).reshape(r, -1, per)
    out = torch.zeros(q.shape[:2], dtype=torch.uint8, device=q.device)
    for i in range(per):
        out |= q[:, :, i] << (i * bits)
    return out


def _weight_parts(k, n, bits, block, zp, dtype, gen):
    """One quantized weight [N, K] as a quantizer leaves normal weights of variance 1/K: values
    spread around their zero points over the whole range, a scale per block, zero points near the
    middle. Returns the values [N, blocks*block] u8, the scales [N, blocks] and the zero points."""
    blocks = -(-k // block)
    mid, top = 1 << (bits - 1), (1 << bits) - 1
    q = torch.randn(n, blocks * block, generator=gen, device=DEVICE)
    q = (q * (top / 6.0) + mid).round_().clamp_(0, top).to(torch.uint8)
    q[:, k:] = 0
    scales = (0.5 + torch.rand(n, blocks, generator=gen, device=DEVICE)) * (6.0 / (top * math.sqrt(k)))
    scales = scales.to(TORCH[dtype])
    zeros = None
    if zp == "packed":
        zeros = (mid + torch.randint(-1, 2, (n, blocks), generator=gen, device=DEVICE)).clamp_(0, top).to(torch.uint8)
    elif zp == "float":
        zeros = (mid + torch.randn(n, blocks, generator=gen, device=DEVICE) * (top / 15.0)).to(TORCH[dtype])
    return q, scales, zeros


def _pack(parts, k, n, bits, block, zp, dtype) -> PackedWeight:
    """The weight packed on the device, as the load-time move keeps it."""
    ctx = _ctx()
    q, scales, zeros = parts
    b = _pack_rows(q, bits)
    z = _pack_rows(zeros, bits) if zp == "packed" else zeros
    kind = {"none": _lib.ZP_NONE, "packed": _lib.ZP_PACKED, "float": _lib.ZP_FLOAT}[zp]
    torch.cuda.synchronize()
    handle = ctypes.c_void_p()
    ctx.check(lib().tmh_weight_pack_nbits(
        ctx.handle, b.data_ptr(), b.numel(), scales.data_ptr(), CODE[dtype], scales.numel(),
        z.data_ptr() if z is not None else None, kind, CODE[dtype] if zp == "float" else _lib.U8,
        z.numel() if z is not None else 0, k, n, bits, block, CODE[dtype], None, ctypes.byref(handle)))
    ctx.synchronize()
    return PackedWeight(ctx, handle, k, n, bits, block, dtype, kind)


def _dense64(parts, k, bits, block, zp):
    """The weight [N, K] in 64 bits."""
    q, scales, zeros = parts
    z = zeros.double() if zeros is not None else torch.full(scales.shape, float(1 << (bits - 1)), dtype=torch.float64,
                                                            device=DEVICE)
    w = (q.reshape(q.shape[0], -1, block).double() - z[:, :, None]) * scales.double()[:, :, None]
    return w.reshape(q.shape[0], -1)[:, :k]


def _merge(a, b):
    return a if a == b else "f32"


def _activations(m, k, dtype, gen):
    """Activations after a norm: unit variance, with a few large channels."""
    x = torch.randn(m, k, generator=gen, device=DEVICE)
    return (x * (1.0 + 4.0 * (torch.rand(k, generator=gen, device=DEVICE) < 0.01))).to(TORCH[dtype])


class _Graph:
    """An executable HIP graph of the calls `body` makes on the context's stream."""

    def __init__(self, ctx, body):
        body()  # sizes the workspace before the capture
        ctx.synchronize()
        self.ctx, self.handle = ctx, ctypes.c_void_p()
        ctx.check(lib().tmh_graph_begin(ctx.handle, None))
        body()
        ctx.check(lib().tmh_graph_end(ctx.handle, None, ctypes.byref(self.handle)))

    def __del__(self):
        if self.handle:
            lib().tmh_graph_destroy(self.ctx.handle, self.handle)


# ---------------------------------------------------------------- op and layers


def _projections(case):
    """(input, K, N) of each MatMulNBits of one layer; inputs are hidden, attention and MLP rows."""
    if case["kind"] == "op":
        return [(0, case["k"], case["n"])]
    h, q, kv, inter = case["hidden"], case["q"], case["kv"], case["inter"]
    return [(0, h, q + 2 * kv), (1, q, h), (0, h, 2 * inter), (2, inter, h)]


def _matmul_inputs(case, seed):
    ks = {i: k for i, k, _n in _projections(case)}
    return {i: _activations(case["m"], k, case["dtype"], _gen(seed, 1, i)) for i, k in ks.items()}


def _matmul_parts(case, seed, layer, p, k, n):
    return _weight_parts(k, n, case["bits"], case["block"], case["zp"], case["weights"], _gen(seed, 2, layer, p))


def _bias(case, seed, n):
    if not case.get("bias"):
        return None
    return torch.randn(n, generator=_gen(seed, 3), device=DEVICE).to(TORCH[_merge(case["dtype"], case["weights"])])


def _prepare_matmul(case, seed):
    ctx = _ctx()
    m, layers = case["m"], case.get("layers", 1)
    inputs = _matmul_inputs(case, seed)
    y_type = _merge(case["dtype"], case["weights"])
    outputs, weights, calls = [], [], []
    for p, (i, k, n) in enumerate(_projections(case)):
        y = torch.empty(layers, m, n, dtype=TORCH[y_type], device=DEVICE)
        bias = _bias(case, seed, n)
        outputs.append(y)
        inputs[("bias", p)] = bias
        for layer in range(layers):
            w = _pack(_matmul_parts(case, seed, layer, p, k, n), k, n, case["bits"], case["block"], case["zp"],
                      case["weights"])
            weights.append(w)
            calls.append((layer, (ctx.handle, w.handle, inputs[i].data_ptr(), CODE[case["dtype"]], m, k,
                                  bias.data_ptr() if bias is not None else None, CODE[y_type] if bias is not None else 0,
                                  y[layer].data_ptr(), CODE[y_type], n, None)))
    calls = [args for _layer, args in sorted(calls, key=lambda c: c[0])]
    state = {"ctx": ctx, "keep": (inputs, weights), "calls": calls, "outputs": outputs, "graph": None}
    if case.get("graph"):
        state["graph"] = _Graph(ctx, lambda: _call_all(ctx, calls))
    return state


def _call_all(ctx, calls):
    matmul = lib().tmh_matmul_nbits
    for args in calls:
        ctx.check(matmul(*args))


def _run_matmul(state):
    if state["graph"] is not None:
        state["ctx"].check(lib().tmh_graph_launch(state["ctx"].handle, state["graph"].handle, None))
    else:
        _call_all(state["ctx"], state["calls"])
    return state["outputs"]


def _exact_matmul(case, seed):
    inputs = _matmul_inputs(case, seed)
    out = []
    for p, (i, k, n) in enumerate(_projections(case)):
        bias = _bias(case, seed, n)
        rows = []
        for layer in range(case.get("layers", 1)):
            w = _dense64(_matmul_parts(case, seed, layer, p, k, n), k, case["bits"], case["block"], case["zp"])
            y = inputs[i].double() @ w.T
            rows.append(y + bias.double() if bias is not None else y)
        out.append(torch.stack(rows))
    return out


def _weight_bytes(k, n, bits, block, zp, dtype):
    blocks = -(-k // block)
    zero = {"none": 0, "packed": n * -(-blocks * bits // 8), "float": n * blocks * SIZE[dtype]}[zp]
    return n * k * bits / 8 + n * blocks * SIZE[dtype] + zero


def _work_matmul(case):
    m, layers, y = case["m"], case.get("layers", 1), SIZE[_merge(case["dtype"], case["weights"])]
    total, flops = 0.0, 0.0
    for _i, k, n in _projections(case):
        total += layers * (_weight_bytes(k, n, case["bits"], case["block"], case["zp"], case["weights"]) + m * n * y)
        total += n * y if case.get("bias") else 0
        flops += layers * 2.0 * m * n * k
    total += sum(m * k * SIZE[case["dtype"]] for k in {i: k for i, k, _n in _projections(case)}.values())
    return {"bytes": total, "flops": flops}


# ---------------------------------------------------------------- vocab


def _vocab_inputs(case, seed):
    parts = _weight_parts(case["dim"], case["rows"], case["bits"], case["block"], "packed", case["dtype"], _gen(seed, 4))
    # Token ids: frequent ones first, as a tokenizer numbers them.
    u = torch.rand(case["ids"], generator=_gen(seed, 5), device=DEVICE, dtype=torch.float64)
    ids = (torch.exp(u * math.log(case["rows"])) - 1).long().clamp_(0, case["rows"] - 1)
    return parts, ids, _activations(case["m"], case["dim"], case["dtype"], _gen(seed, 6))


def _prepare_vocab(case, seed):
    ctx = _ctx()
    rows, dim, bits, block, dtype = case["rows"], case["dim"], case["bits"], case["block"], case["dtype"]
    parts, ids, x = _vocab_inputs(case, seed)
    w = _pack(parts, dim, rows, bits, block, "packed", dtype)
    data, scales, zeros = _pack_rows(parts[0], bits), parts[1], _pack_rows(parts[2], bits)
    embedded = torch.empty(case["ids"], dim, dtype=TORCH[dtype], device=DEVICE)
    logits = torch.empty(case["m"], rows, dtype=TORCH[dtype], device=DEVICE)
    gather = (ctx.handle, data.data_ptr(), _lib.U8, rows, data.shape[1], ids.data_ptr(), _lib.S64, case["ids"],
              scales.data_ptr(), CODE[dtype], scales.shape[1], zeros.data_ptr(), _lib.U8, bits, embedded.data_ptr(), None)
    head = (ctx.handle, w.handle, x.data_ptr(), CODE[dtype], case["m"], dim, None, 0, logits.data_ptr(), CODE[dtype],
            rows, None)
    return {"ctx": ctx, "keep": (w, data, scales, zeros, ids, x), "gather": gather, "head": head,
            "outputs": {"embedded": embedded, "logits": logits}}


def _run_vocab(state):
    ctx = state["ctx"]
    ctx.check(lib().tmh_gather_block_quantized(*state["gather"]))
    ctx.check(lib().tmh_matmul_nbits(*state["head"]))
    return state["outputs"]


def _exact_vocab(case, seed):
    parts, ids, x = _vocab_inputs(case, seed)
    w = _dense64(parts, case["dim"], case["bits"], case["block"], "packed")
    return {"embedded": w[ids], "logits": x.double() @ w.T}


def _work_vocab(case):
    size, row = SIZE[case["dtype"]], _weight_bytes(case["dim"], 1, case["bits"], case["block"], "packed", case["dtype"])
    total = case["rows"] * (row + case["m"] * size) + case["m"] * case["dim"] * size
    total += case["ids"] * (8 + row + case["dim"] * size)
    return {"bytes": total, "flops": 2.0 * case["m"] * case["rows"] * case["dim"]}


# ---------------------------------------------------------------- qmoe


def _expert_shapes(case):
    shapes = [(case["inter"], case["hidden"]), (case["hidden"], case["inter"])]  # fc1, fc2
    return shapes + [(case["inter"], case["hidden"])] if case["activation"] == "swiglu" else shapes  # fc3


def _expert_parts(case, seed, i):
    n, k = _expert_shapes(case)[i]
    return _weight_parts(k, case["experts"] * n, case["bits"], case["block"], "none", case["dtype"], _gen(seed, 7, i))


def _qmoe_inputs(case, seed):
    x = _activations(case["tokens"], case["hidden"], case["dtype"], _gen(seed, 8))
    router = torch.randn(case["tokens"], case["experts"], generator=_gen(seed, 9), device=DEVICE)
    return x, router


def _prepare_qmoe(case, seed):
    ctx = _ctx()
    experts, bits, block, dtype = case["experts"], case["bits"], case["block"], case["dtype"]
    weights = []
    for i, (n, k) in enumerate(_expert_shapes(case)):
        q, scales, _zeros = _expert_parts(case, seed, i)
        packed = _pack_rows(q[:, :k], bits).reshape(experts, n, -1).cpu().numpy()
        weights.append(ExpertWeight.upload(ctx, packed, scales.reshape(experts, n, -1).cpu().numpy(), None, bits=bits,
                                           block_size=block, dtype=dtype))
    fc1, fc2, fc3 = (weights + [None])[:3]
    x, router = _qmoe_inputs(case, seed)
    y = torch.empty_like(x)
    args = (ctx.handle, x.data_ptr(), CODE[dtype], case["tokens"], case["hidden"], router.data_ptr(), _lib.F32, experts,
            case["k"], fc1.handle, None, fc2.handle, None, fc3.handle if fc3 else None, None, CODE[dtype],
            _lib.ACTIVATIONS[case["activation"]], 0, 1.0, 0.0, 0.0, y.data_ptr(), None)
    torch.cuda.synchronize()
    return {"ctx": ctx, "keep": (weights, x, router), "args": args, "outputs": y}


def _run_qmoe(state):
    state["ctx"].check(lib().tmh_qmoe(*state["args"]))
    return state["outputs"]


def _exact_qmoe(case, seed):
    x, router = _qmoe_inputs(case, seed)
    x = x.double()
    top, index = torch.topk(router.double(), case["k"], dim=1)
    gate = torch.softmax(top, dim=1)
    dense = [_dense64(_expert_parts(case, seed, i), k, case["bits"], case["block"], "none").reshape(case["experts"], n, k)
             for i, (n, k) in enumerate(_expert_shapes(case))]
    y = torch.zeros_like(x)
    for e in range(case["experts"]):
        rows, slots = torch.nonzero(index == e, as_tuple=True)
        if not len(rows):
            continue
        h = x[rows] @ dense[0][e].T
        if case["activation"] == "swiglu":
            h = h * torch.sigmoid(h) * (x[rows] @ dense[2][e].T)
        elif case["activation"] == "silu":
            h = h * torch.sigmoid(h)
        else:
            h = 0.5 * h * (1 + torch.erf(h / math.sqrt(2)))
        y.index_add_(0, rows, (h @ dense[1][e].T) * gate[rows, slots][:, None])
    return y


def _work_qmoe(case):
    t, e, k, size = case["tokens"], case["experts"], case["k"], SIZE[case["dtype"]]
    used = e * (1 - (1 - k / e) ** t)  # experts that at least one token takes, on average
    per = sum(_weight_bytes(kk, n, case["bits"], case["block"], "none", case["dtype"]) for n, kk in _expert_shapes(case))
    flops = 2.0 * t * k * sum(n * kk for n, kk in _expert_shapes(case))
    return {"bytes": used * per + 2 * t * case["hidden"] * size + 4 * t * e, "flops": flops}


# ---------------------------------------------------------------- int8


def _int8_inputs(case, seed):
    m, k, n = case["m"], case["k"], case["n"]
    x = torch.randn(m, k, generator=_gen(seed, 10), device=DEVICE)
    gen = _gen(seed, 11)
    b = (torch.randn(k, n, generator=gen, device=DEVICE) * 32).round_().clamp_(-127, 127).to(torch.int8)
    if case["b"] == "u8":
        b = (b.int() + 128).to(torch.uint8)
    z = None
    if case["b_zero"]:
        z = torch.randint(-3, 4, (n,), generator=gen, device=DEVICE)
        z = (z + 128).to(torch.uint8) if case["b"] == "u8" else z.to(torch.int8)
    return x, b, z, (0.5 + torch.rand(n, generator=gen, device=DEVICE)) * 1e-3


def _prepare_int8(case, seed):
    ctx = _ctx()
    m, k, n = case["m"], case["k"], case["n"]
    x, b, z, scales = _int8_inputs(case, seed)
    torch.cuda.synchronize()
    handle = ctypes.c_void_p()
    ctx.check(lib().tmh_int8_weight_prepare(ctx.handle, b.data_ptr(), _lib.U8 if case["b"] == "u8" else _lib.S8,
                                            z.data_ptr() if z is not None else None, n if z is not None else 0, k, n,
                                            None, ctypes.byref(handle)))
    ctx.synchronize()
    w = Int8Weight(ctx, handle, k, n, case["b"])
    q = torch.empty(m, k, dtype=torch.uint8, device=DEVICE)
    scale = torch.empty((), dtype=torch.float32, device=DEVICE)
    zero = torch.empty((), dtype=torch.uint8, device=DEVICE)
    sums = torch.empty(m, n, dtype=torch.int32, device=DEVICE)
    y = torch.empty(m, n, dtype=torch.float32, device=DEVICE)
    quantize = (ctx.handle, x.data_ptr(), _lib.F32, x.numel(), q.data_ptr(), scale.data_ptr(), zero.data_ptr(), None)
    product = (ctx.handle, q.data_ptr(), _lib.U8, zero.data_ptr(), 1, 1, m, w.handle, sums.data_ptr(), None)
    dequantize = (ctx.handle, sums.data_ptr(), _lib.S32, m, n, 1, scales.data_ptr(), _lib.F32, None, 0,
                  _lib.QPARAM_AXIS, 0, y.data_ptr(), None)
    return {"ctx": ctx, "keep": (w, x, scales), "quantize": quantize, "product": product, "dequantize": dequantize,
            "outputs": {"q": q, "scale": scale, "zero": zero, "sums": sums, "y": y}}


def _run_int8(state):
    ctx = state["ctx"]
    ctx.check(lib().tmh_dynamic_quantize_linear(*state["quantize"]))
    ctx.check(lib().tmh_matmul_integer_prepared(*state["product"]))
    ctx.check(lib().tmh_dequantize_linear(*state["dequantize"]))
    return state["outputs"]


def _exact_int8(case, seed):
    x, b, z, scales = _int8_inputs(case, seed)
    # The quantization is defined by its f32 steps: whole values follow from them exactly.
    low, high = x.min().clamp(max=0), x.max().clamp(min=0)
    scale = (high - low) / 255
    zero = torch.round(-low / scale).clamp(0, 255)
    q = (torch.round(x / scale) + zero).clamp(0, 255)
    bz = z.double() if z is not None else torch.zeros(case["n"], dtype=torch.float64, device=DEVICE)
    sums = (q.double() - zero.double()) @ (b.double() - bz)
    return {"q": q.to(torch.uint8), "scale": scale, "zero": zero.to(torch.uint8), "sums": sums.to(torch.int32),
            "y": sums * scales.double()}


def _work_int8(case):
    m, k, n = case["m"], case["k"], case["n"]
    return {"bytes": 4.0 * m * k + 2.0 * m * k + k * n + 3 * 4.0 * m * n + 8.0 * n, "flops": 2.0 * m * k * n}


# ---------------------------------------------------------------- the interface

_KINDS = {
    "op": (_prepare_matmul, _run_matmul, _exact_matmul, _work_matmul),
    "layers": (_prepare_matmul, _run_matmul, _exact_matmul, _work_matmul),
    "vocab": (_prepare_vocab, _run_vocab, _exact_vocab, _work_vocab),
    "qmoe": (_prepare_qmoe, _run_qmoe, _exact_qmoe, _work_qmoe),
    "int8": (_prepare_int8, _run_int8, _exact_int8, _work_int8),
}


def prepare(case, seed):
    state = _KINDS[case["kind"]][0](case, seed)
    torch.cuda.synchronize()
    state["run"] = _KINDS[case["kind"]][1]
    return state


def run(state):
    return state["run"](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    # About four times the largest error against exact() that the cases and their draws show: the
    # type of Y, the rounding of the weights to their own type and (f32, over 64 rows) the 16 bits
    # that the prefill keeps of each factor.
    if case["kind"] == "int8":
        return "exact"  # whole numbers, and one f32 product of each
    if case["kind"] == "qmoe":
        return {"rel": 3.5e-3, "max": 4e-2}  # every intermediate rounds to f16
    return {"f16": {"rel": 1.2e-3, "max": 6e-3}, "bf16": {"rel": 9e-3, "max": 5e-2},
            "f32": {"rel": 2e-5, "max": 2e-4}}[_merge(case["dtype"], case.get("weights", case["dtype"]))]
