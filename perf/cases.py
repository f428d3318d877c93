"""The calls this package is measured on: the matmul path of a Qwen3-4B engine (hidden 2,560,
intermediate 9,728, QKV 6,144, attention output 4,096, vocabulary 151,936) as an engine makes them.

  call    one projection of one layer, called eagerly: the smallest call, all latency
  decode  a decode step's projections (QKV, O, gate_up with SwiGLU, down) over several layers of
          distinct weights, captured in a graph as an engine's decode step is: 1 row is plain
          decoding, 2 to 16 rows batched decoding, up to 32 rows batched tree verification
  fused   the same with the residual adds and RMSNorms folded into the projections
  head    the lm head with greedy argmax
  prefill the projections of one layer over a prompt, called eagerly: short prompts (chat turns), odd
          lengths, and one chunk of a long prompt
  load    the weight quantization of one layer, as at engine load

Each returns every output of its projections. A layer's weights are 101 MB in FP8, so the graphs
over several layers read their weights from HBM, as a 36-layer engine does.
"""

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "kernel-rush-qwen_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

H, I, NQKV, NQD, V = 2560, 9728, 6144, 4096, 151936
SHAPES = {"qkv": (NQKV, H), "o": (H, NQD), "gate_up": (2 * I, H), "down": (H, I)}
# the engine's output contract: fp32 split-K partials for QKV, O and down, SwiGLU for gate_up
SPLIT = {"qkv": 2, "o": 4, "down": 4}
EPS = 1e-6
FP8_LAYERS, BF16_LAYERS = 8, 4  # about 0.8 GB of weights each, several times the last-level cache


def listed():
    return [
        # one attention-output projection of a decode step, outside a graph
        {"name": "call_o_m1", "op": "call", "proj": "o", "rows": 1},
        # greedy decoding of one sequence, FP8 weights
        {"name": "decode_fp8_m1", "op": "decode", "weights": "fp8", "scale": "token", "rows": 1},
        # a small odd batch
        {"name": "decode_fp8_m5", "op": "decode", "weights": "fp8", "scale": "token", "rows": 5},
        # batch 16
        {"name": "decode_fp8_m16", "op": "decode", "weights": "fp8", "scale": "token", "rows": 16},
        # batch 16 with two verify rows each, activation scales calibrated at prefill
        {"name": "decode_fp8_m32_static", "op": "decode", "weights": "fp8", "scale": "static", "rows": 32},
        # greedy decoding and batch 16 on the checkpoint's own BF16 weights (the engine's default)
        {"name": "decode_bf16_m1", "op": "decode", "weights": "bf16", "packed": False, "rows": 1},
        {"name": "decode_bf16_m16", "op": "decode", "weights": "bf16", "packed": False, "rows": 16},
        # the fused decoder layer at batch 16
        {"name": "fused_fp8_m16", "op": "fused", "rows": 16},
        # the FP8 lm head at batch 16
        {"name": "head_fp8_m16", "op": "head", "weights": "fp8", "rows": 16},
        # a chat turn of 77 tokens, and a 4,096-token chunk of a long prompt
        {"name": "prefill_77", "op": "prefill", "scale": "tensor", "rows": 77},
        {"name": "prefill_4096", "op": "prefill", "scale": "tensor", "rows": 4096},
        # one layer's weights quantized per output channel
        {"name": "load_channel", "op": "load", "scale": "channel"},
    ]


def draw(rng):
    plain = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    case = _draw(rng)
    while case in plain:
        case = _draw(rng)
    return case


def _draw(rng):
    rows = rng.randint(1, 32)
    op = rng.choice(["call", "decode", "decode", "decode", "fused", "head", "prefill", "prefill", "load"])
    if op == "call":
        return {"op": op, "proj": rng.choice(sorted(SHAPES)), "rows": rows}
    if op == "decode":
        if rng.random() < 0.6:
            return {"op": op, "weights": "fp8", "scale": rng.choice(["token", "static"]), "rows": rows}
        return {"op": op, "weights": "bf16", "packed": rng.choice([False, True]), "rows": rows}
    if op == "fused":
        return {"op": op, "rows": rows}
    if op == "head":
        return {"op": op, "weights": rng.choice(["fp8", "bf16"]), "rows": rows}
    if op == "prefill":
        rows = int(round(math.exp(rng.uniform(math.log(33), math.log(4096)))))
        return {"op": op, "scale": rng.choice(["tensor", "static"]), "rows": rows}
    # the layer's weights, or one shard's rows of them (tensor-parallel degree 1 to 8, 16-row blocks)
    return {"op": op, "scale": rng.choice(["channel", "tensor"]), "rows_of_shard": 16 * rng.randint(20, 160)}


# ----------------------------------------------------------------------------------------------
# inputs: weights N(0, 0.02), activations N(0, 1) with the heavier-tailed SwiGLU products in front
# of the down projection, as the layers of a trained model show them
# ----------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.bfloat16)


def _weight(g, name):
    return _randn(g, *SHAPES[name]).mul_(0.02)


def _acts(g, rows):
    x = {"qkv": _randn(g, rows, H), "o": _randn(g, rows, NQD), "gate_up": _randn(g, rows, H)}
    x["down"] = torch.nn.functional.silu(_randn(g, rows, I)) * _randn(g, rows, I)
    return x


def _layers(case):
    return BF16_LAYERS if case.get("weights") == "bf16" else FP8_LAYERS


def _inputs(case, seed):
    """Every input tensor of the case, from the seed alone."""
    g, op = _gen(seed), case["op"]
    if op == "call":
        return {"w": _weight(g, case["proj"]), "x": _acts(g, case["rows"])[case["proj"]]}
    if op == "load":
        if "rows_of_shard" in case:
            return {n: _weight(g, n)[:case["rows_of_shard"]].contiguous() for n in SHAPES}
        return {n: _weight(g, n) for n in SHAPES}
    if op == "prefill":
        return {"w": {n: _weight(g, n) for n in SHAPES}, "x": _acts(g, case["rows"])}
    if op == "head":
        e = _randn(g, V, H).mul_(0.02)
        ids = torch.randint(0, V, (case["rows"],), generator=g, device="cuda")
        # hidden states that favour one token clearly, as a trained model's do
        h = (_randn(g, case["rows"], H) + e[ids] * 20).to(torch.bfloat16)
        return {"w": e, "x": h}
    out = []
    for _ in range(_layers(case)):
        d = {"w": {n: _weight(g, n) for n in SHAPES}, "x": _acts(g, case["rows"])}
        if op == "fused":
            d["res"] = _randn(g, case["rows"], H)
            d["ln"] = [(1 + 0.1 * _randn(g, H)).to(torch.bfloat16) for _ in range(2)]
        out.append(d)
    return out


# ----------------------------------------------------------------------------------------------
# the framework's calls
# ----------------------------------------------------------------------------------------------
def _shared(x):
    from kernels import fp8
    a = fp8.ActScale(x, headroom=2.0)
    return fp8.SharedScale(a.inv, a.scale)


def _graph(step):
    """The step captured as an engine captures its decode step: (graph, its output buffers)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return {"graph": graph, "out": out}


def _decode_fp8(layers):
    from kernels import fp8

    def step():
        out = []
        for d in layers:
            q, x, a = d["q"], d["x"], d["a"]
            act = fp8.gemv_swiglu_fp8(x["gate_up"], q["gate_up"], a=a["gate_up"])
            out.append({"qkv": fp8.gemv_fp8(x["qkv"], q["qkv"], SPLIT["qkv"], a=a["qkv"]),
                        "o": fp8.gemv_fp8(x["o"], q["o"], SPLIT["o"], a=a["o"]), "act": act,
                        "down": fp8.gemv_fp8(act, q["down"], SPLIT["down"], a=a["down"])})
        return out
    return step


def _decode_bf16(layers):
    from kernels.gemv import gemv, gemv_swiglu

    def step():
        out = []
        for d in layers:
            w, x = d["w"], d["x"]
            act = gemv_swiglu(x["gate_up"], w["gate_up"])
            out.append({"qkv": gemv(x["qkv"], w["qkv"], SPLIT["qkv"]), "o": gemv(x["o"], w["o"], SPLIT["o"]),
                        "act": act, "down": gemv(act, w["down"], SPLIT["down"])})
        return out
    return step


def _fused_fp8(layers, rows):
    from kernels.fused_gemv import FusedLayerBuffers, gemv_fused, gemv_swiglu_fused
    bufs = [FusedLayerBuffers(rows, H, V, "cuda") for _ in layers]

    def step():
        out = []
        for d, b in zip(layers, bufs):
            q, ln = d["q"], d["ln"]
            gemv_fused(d["x"]["o"], q["o"], SPLIT["o"], ep=(d["res"], b.res[1], b.ss[1], b.cnt), eps=EPS)
            act = gemv_swiglu_fused(b.res[1], q["gate_up"], norm=(ln[1], b.ss[1]), eps=EPS)
            gemv_fused(act, q["down"], SPLIT["down"], ep=(b.res[1], b.res[0], b.ss[0], b.cnt), eps=EPS)
            qkv = gemv_fused(b.res[0], q["qkv"], SPLIT["qkv"], norm=(ln[0], b.ss[0]), eps=EPS)
            out.append({"mid": b.res[1], "act": act, "res": b.res[0], "qkv": qkv})
        return out
    return step


def prepare(case, seed):
    from kernels import fp8
    from kernels.gemv import pack
    op, d = case["op"], _inputs(case, seed)
    if op == "call":
        return {"op": op, "q": fp8.quantize(d["w"]), "x": d["x"], "split": SPLIT.get(case["proj"])}
    if op == "load":
        return {"op": op, "w": d, "fn": fp8.quantize if case["scale"] == "channel" else fp8.quantize_weight}
    if op == "prefill":
        static = case["scale"] == "static"
        return {"op": op, "q": {n: fp8.quantize_weight(w) for n, w in d["w"].items()}, "x": d["x"],
                "a": {n: _shared(x) if static else None for n, x in d["x"].items()}}
    if op == "head":
        return {"op": op, "w": fp8.quantize(d["w"]) if case["weights"] == "fp8" else pack(d["w"]), "x": d["x"]}
    for l in d:
        if case.get("weights") == "bf16":
            if case["packed"]:
                l["w"] = {n: pack(w) for n, w in l["w"].items()}
        else:
            l["q"] = {n: fp8.quantize(w) for n, w in l["w"].items()}
            static = case.get("scale") == "static"
            l["a"] = {n: _shared(l["x"][n]) if static else None for n in SHAPES}
            del l["w"]
    if op == "fused":
        step = _fused_fp8(d, case["rows"])
    else:
        step = _decode_bf16(d) if case["weights"] == "bf16" else _decode_fp8(d)
    return {"op": op, "step": step, **_graph(step)}  # (step holds the tensors that the graph reads)


def run(state):
    op = state["op"]
    if op in ("decode", "fused"):
        state["graph"].replay()
        return state["out"]
    from kernels import fp8
    from kernels.lmhead import lm_head_argmax
    if op == "call":
        if state["split"] is None:
            return fp8.gemv_swiglu_fp8(state["x"], state["q"])
        return fp8.gemv_fp8(state["x"], state["q"], state["split"])
    if op == "head":
        return lm_head_argmax(state["x"], state["w"], return_logits=True)
    if op == "prefill":
        return {n: fp8.linear_fp8(state["x"][n], state["q"][n], state["a"][n]) for n in SHAPES}
    out = {}
    for n, w in state["w"].items():
        q = state["fn"](w)
        out[n] = {"w8": q[0].view(torch.uint8), "scale": q[1], "tiled": q.tiled}
    return out


# ----------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------
def _proj_work(name, rows, wbytes, split=None):
    """Weights (with their scales, in FP8) and activations read once, the output written once."""
    n, k = SHAPES[name]
    out = 2 * rows * I if name == "gate_up" else 4 * split * rows * n if split else 2 * rows * n
    scales = 4 * n if wbytes == 1 else 0
    return n * k * wbytes + scales + 2 * rows * k + out, 2 * rows * n * k


def work(case):
    op, rows = case["op"], case.get("rows", 0)
    if op == "call":
        b, f = _proj_work(case["proj"], rows, 1, SPLIT.get(case["proj"]))
    elif op == "load":
        m = {n: (case.get("rows_of_shard") or s[0]) for n, s in SHAPES.items()}
        # bf16 in; the e4m3 bytes out in both layouts, and the scales
        b = sum(m[n] * s[1] * 4 + (4 * m[n] if case["scale"] == "channel" else 4) for n, s in SHAPES.items())
        f = sum(2 * m[n] * s[1] for n, s in SHAPES.items())
    elif op == "prefill":
        b = sum(n * k + 4 + 2 * rows * k + 2 * rows * n for n, k in SHAPES.values())
        f = sum(2 * rows * n * k for n, k in SHAPES.values())
    elif op == "head":
        wb = 1 if case["weights"] == "fp8" else 2
        b = V * H * wb + (4 * V if wb == 1 else 0) + 2 * rows * H + 2 * rows * V + 8 * rows
        f = 2 * rows * V * H
    else:
        wb = 2 if case.get("weights") == "bf16" else 1
        b = f = 0
        for n in SHAPES:
            split = None if op == "fused" and n != "qkv" else SPLIT.get(n)
            pb, pf = _proj_work(n, rows, wb, split)
            if op == "fused":  # the residual rows read, or the RMSNorm weight
                pb += 2 * rows * H if n in ("o", "down") else 2 * H
            b, f = b + pb, f + pf
        b, f = b * _layers(case), f * _layers(case)
    return {"bytes": b, "flops": f}


def tolerance(case):
    op = case["op"]
    if op == "load":
        return "exact"
    # bf16 results, 1.7e-3 off the 64-bit sums
    if op == "prefill":
        return {"rel": 4e-3, "max": 0.03}
    if op == "head":
        return {"rel": 4e-3, "max": 0.03, "differ": 0.0}
    # bf16 activations that are rounded to e4m3 again: a value on the other side of one bf16 rounding
    # moves an e4m3 code. Against 64 bits: down after SwiGLU 2e-3, and in the fused layer, where the
    # residual row passes two norms, up to 1.5e-2 in QKV
    return {"rel": 3e-2, "max": 0.75} if op == "fused" else {"rel": 1e-2, "max": 0.25}


# ----------------------------------------------------------------------------------------------
# the same results from plain torch, with every sum in 64 bits: the roundings that define the path
# (e4m3 operands and their fp32 scales, bf16 activations between projections) are kept
# ----------------------------------------------------------------------------------------------
INV448 = torch.tensor(1.0, dtype=torch.float32) / torch.tensor(448.0, dtype=torch.float32)


def _e4m3(v):
    return v.clamp(-448.0, 448.0).to(torch.float8_e4m3fn)


def _quant_w(w, per_tensor=False):
    """(e4m3 bytes' values in fp32, fp32 scale, e4m3 tensor) of a weight."""
    wf = w.float()
    amax = wf.abs().amax() if per_tensor else wf.abs().amax(1, keepdim=True)
    scale = amax.clamp_min(1e-12) * INV448.to(w.device)
    w8 = _e4m3(wf / scale)
    return w8, scale


def _quant_x(x, mode):
    """(values, scale) of activations: per token, per tensor, or per tensor with headroom 2."""
    xf = x.float()
    amax = xf.abs().amax(1, keepdim=True) if mode == "token" else xf.abs().amax()
    amax = amax.clamp_min(1e-6) * (2.0 if mode == "static" else 1.0)
    return _e4m3(xf * (amax.reciprocal() * 448.0)), amax * INV448.to(x.device)


def _mul64(a, b, sa=None, sb=None):
    """a @ b.T in fp64, in slices of b's rows; scales applied in fp64."""
    a = a.double()
    out = torch.cat([a @ c.double().t() for c in b.split(8192)], 1)
    if sa is not None:
        out = out * sa.double() * sb.double().reshape(1, -1)
    return out


def _split64(x, w, split, sx=None, sw=None):
    k = x.shape[1] // split
    return torch.stack([_mul64(x[:, s * k:(s + 1) * k], w[:, s * k:(s + 1) * k], sx, sw) for s in range(split)])


def _bf(t):
    return t.to(torch.bfloat16)


def _swiglu64(gu):
    g, u = _bf(gu[:, :I]).double(), _bf(gu[:, I:]).double()
    return _bf(g / (1 + torch.exp(-g))).double() * u


def _lin64(x, w, mode, split=None, a_of=None):
    """x @ w.T of the FP8 path in fp64 (w quantized per output channel)."""
    w8, sw = _quant_w(w)
    if mode == "static":
        amax = (x if a_of is None else a_of).float().abs().amax().clamp_min(1e-6) * 2.0
        x8, sx = _e4m3(x.float() * (amax.reciprocal() * 448.0)), amax * INV448.to(x.device)
    else:
        x8, sx = _quant_x(x, "token")
    x8, w8 = x8.float(), w8.float()
    return _split64(x8, w8, split, sx, sw) if split else _mul64(x8, w8, sx, sw)


def _rms64(x, ln):
    xd = x.double()
    h = _bf(xd * torch.rsqrt(xd.pow(2).mean(1, keepdim=True) + EPS))
    return _bf(h.double() * ln.double())


def exact(case, seed):
    op, d = case["op"], _inputs(case, seed)
    if op == "load":
        out = {}
        for n, w in d.items():
            w8, s = _quant_w(w, case["scale"] == "tensor")
            out[n] = {"w8": w8.view(torch.uint8), "scale": s.reshape(-1).double() if s.dim() else s.double(),
                      "tiled": None}
        return out
    if op == "call":
        if case["proj"] == "gate_up":
            return _swiglu64(_lin64(d["x"], d["w"], "token"))
        return _lin64(d["x"], d["w"], "token", SPLIT[case["proj"]])
    if op == "head":
        logits = _lin64(d["x"], d["w"], "token") if case["weights"] == "fp8" else _mul64(d["x"], d["w"])
        return torch.argmax(logits, -1), logits
    if op == "prefill":
        out = {}
        for n, w in d["w"].items():
            w8, sw = _quant_w(w, True)
            x8, sx = _quant_x(d["x"][n], case["scale"])
            out[n] = _mul64(x8.float(), w8.float(), sx, sw)
        return out
    out = []
    for l in d:
        w, x = l["w"], l["x"]
        if op == "fused":
            mid = _bf(l["res"].double() + _bf(_lin64(x["o"], w["o"], "token")).double())
            act = _swiglu64(_lin64(_rms64(mid, l["ln"][1]), w["gate_up"], "token"))
            res = _bf(mid.double() + _bf(_lin64(_bf(act), w["down"], "token")).double())
            qkv = _lin64(_rms64(res, l["ln"][0]), w["qkv"], "token", SPLIT["qkv"])
            out.append({"mid": mid.double(), "act": act, "res": res.double(), "qkv": qkv})
        elif case["weights"] == "bf16":
            act = _swiglu64(_mul64(x["gate_up"], w["gate_up"]))
            out.append({"qkv": _split64(x["qkv"], w["qkv"], SPLIT["qkv"]), "o": _split64(x["o"], w["o"], SPLIT["o"]),
                        "act": act, "down": _split64(_bf(act), w["down"], SPLIT["down"])})
        else:
            m = case["scale"]
            act = _swiglu64(_lin64(x["gate_up"], w["gate_up"], m))
            out.append({"qkv": _lin64(x["qkv"], w["qkv"], m, SPLIT["qkv"]),
                        "o": _lin64(x["o"], w["o"], m, SPLIT["o"]), "act": act,
                        "down": _lin64(_bf(act), w["down"], m, SPLIT["down"], a_of=x["down"])})
    return out
