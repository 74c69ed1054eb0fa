"""The calls whose speed counts, as data: what a sam3.c program asks of this
backend, through the entry points it would call.

`listed()` names twelve of them, `draw(rng)` makes more of the same kinds over
the whole range of sizes. `prepare` sets up what such a program holds before
the call (weights in HBM, a backend, device buffers), `run` is one pass,
`exact` the same result in float64 with plain torch.

Kinds:
  text      text-encoder layers through graph_eval (Q8_0 weights)
  vit       one ViT image-encoder block through graph_eval
  neck      the FPN neck's scales through graph_eval (f32 convolutions)
  linear    one dense bf16 / f16 linear layer, device pointers
  q8        one Q8_0 linear layer, device pointers
  q8batch   a stream of Q8_0 layers in one call
  sdpa      fused attention, device pointers
  attn      the attention matmuls on their own (Q K^T, P V), device pointers
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

# the package lies in a folder whose name is no module name
sys.path.insert(0, os.path.join(os.getcwd(), "sam3.c_amd"))

from sam3_amd import abi, graph, hip  # noqa: E402

DEV = "cuda"
DT = {"f32": abi.F32, "bf16": abi.BF16, "f16": abi.F16}
TT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
HEAD = 64  # head size of both encoders


def listed():
    return [
        # one token's worth of text encoder (width 1024, 16 heads): the launch-bound end
        {"name": "text_token", "kind": "text", "seq": 1, "width": 1024, "layers": 4},
        # a whole text prompt through the same layers
        {"name": "text_prompt", "kind": "text", "seq": 32, "width": 1024, "layers": 4},
        # prompt decoder: a few rows against a stream of distinct Q8_0 weights
        {"name": "q8_stream_rows8", "kind": "q8batch", "copies": 24, "m": 8, "n": 4096, "k": 1024},
        # one Q8_0 projection of an image's tokens, f32 activations, weights new to each call
        {"name": "q8_linear_image", "kind": "q8", "m": 5184, "n": 1024, "k": 1024, "a": "f32"},
        # ViT-L MLP fc1 on one image, bias and GELU in the epilogue
        {"name": "bf16_fc1_gelu", "kind": "linear", "dtype": "bf16", "m": 5184, "n": 4096,
         "k": 1024, "bias": True, "gelu": True, "nt": True},
        # a ragged f16 layer: a cropped image's tokens, sizes that divide by no tile
        {"name": "f16_ragged", "kind": "linear", "dtype": "f16", "m": 1369, "n": 1000, "k": 1544,
         "bias": True, "gelu": False, "nt": True},
        # windowed ViT attention, 81 windows of 24x24 tokens x 16 heads
        {"name": "sdpa_bf16_windows", "kind": "sdpa", "dtype": "bf16", "bh": 1296, "sq": 576,
         "sk": 576, "mask": False},
        # f32 attention over an odd token count (37x37) with an additive mask
        {"name": "sdpa_f32_masked", "kind": "sdpa", "dtype": "f32", "bh": 16, "sq": 1369,
         "sk": 1369, "mask": True},
        # the same windows with scores and probabilities materialized
        {"name": "attn_matmuls_windows", "kind": "attn", "bh": 1296, "s": 576},
        # one windowed image-encoder block of a quantized checkpoint
        {"name": "vit_window_q8", "kind": "vit", "grid": 72, "window": 24, "width": 1024,
         "global": False, "weights": "q8"},
        # one global-attention block of an f32 checkpoint
        {"name": "vit_global_f32", "kind": "vit", "grid": 72, "window": 24, "width": 1024,
         "global": True, "weights": "f32"},
        # the neck on the trunk's 72x72 map: transposed, 1x1 and 3x3 convolutions, pooling
        {"name": "neck_f32", "kind": "neck", "grid": 72, "dim": 1024, "d": 256},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["text", "q8batch", "q8", "linear", "sdpa", "attn", "vit", "neck"])
    if kind == "text":
        return {"kind": kind, "seq": _log(rng, 1, 77), "width": rng.choice([512, 768, 1024]),
                "layers": rng.randint(1, 4)}
    if kind == "q8batch":
        return {"kind": kind, "copies": rng.randint(2, 32), "m": _log(rng, 1, 77),
                "n": 8 * _log(rng, 32, 512), "k": 256 * _log(rng, 1, 16)}
    if kind == "q8":
        return {"kind": kind, "m": _log(rng, 1, 5184), "n": 4 * _log(rng, 64, 1024),
                "k": 32 * _log(rng, 8, 128), "a": rng.choice(["f32", "f32", "bf16"])}
    if kind == "linear":
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16"]), "m": _log(rng, 16, 5184),
                "n": 8 * _log(rng, 32, 512), "k": 8 * _log(rng, 32, 512),
                "bias": rng.random() < 0.7, "gelu": rng.random() < 0.4, "nt": rng.random() < 0.8}
    if kind == "sdpa":
        side = rng.randint(7, 40)
        sq = side * side
        sk = sq if rng.random() < 0.7 else _log(rng, 16, 2000)
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16", "f32"]),
                "bh": max(1, min(1296, int(rng.uniform(0.1, 1.0) * 16 * 5184 * 1024 / (sq * sk)))),
                "sq": sq, "sk": sk, "mask": rng.random() < 0.4}
    if kind == "attn":
        side = 4 * rng.randint(2, 8)
        return {"kind": kind, "bh": 16 * rng.randint(1, max(1, int(81 * (24 / side) ** 4)) if side > 24
                                                     else 81), "s": side * side}
    if kind == "vit":
        window = rng.randint(7, 24)
        return {"kind": kind, "grid": window * rng.randint(1, 72 // window), "window": window,
                "width": rng.choice([512, 768, 1024]), "global": rng.random() < 0.3,
                "weights": rng.choice(["q8", "f32"])}
    return {"kind": kind, "grid": 2 * rng.randint(8, 36), "dim": rng.choice([512, 768, 1024]),
            "d": rng.choice([128, 256])}


# ------------------------------------------------------------------ inputs
class _Rand:
    """Named normal tensors on the GPU, made from the seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)

    def __call__(self, *shape, std=1.0, mean=0.0):
        x = torch.randn(*shape, generator=self.g, device=DEV, dtype=torch.float32)
        return x.mul_(std).add_(mean) if (std != 1.0 or mean) else x


def _q8(w):
    """Q8_0 blocks (f32 scale, 32 int8; 36 bytes) of an f32 tensor whose
    size divides by 32, as a flat uint8 tensor."""
    b = w.reshape(-1, 32)
    scale = b.abs().amax(1, keepdim=True) / 127.0
    x = torch.where(scale > 0, b / scale, torch.zeros_like(b))
    q = torch.trunc(x + torch.copysign(torch.full_like(x, 0.5), x)).clamp_(-127, 127)
    out = torch.empty(b.shape[0], 36, dtype=torch.uint8, device=w.device)
    out[:, :4] = scale.contiguous().view(torch.uint8)
    out[:, 4:] = q.to(torch.int8).view(torch.uint8)
    return out.reshape(-1)


def _deq64(blocks, shape):
    b = blocks.reshape(-1, 36)
    scale = b[:, :4].contiguous().view(torch.float32).double()
    return (b[:, 4:].contiguous().view(torch.int8).double() * scale).reshape(shape)


def _layer_params(r, width, wkind):
    """The weights of one encoder layer, [out, in]: (kind, shape, tensor)
    by name; the linear weights Q8_0 blocks when wkind is q8."""
    mlp = 4 * width
    p = {}
    for k, shape in (("qkv_w", (3 * width, width)), ("proj_w", (width, width)),
                     ("fc1_w", (mlp, width)), ("fc2_w", (width, mlp))):
        w = r(*shape, std=0.02)
        p[k] = ("q8", shape, _q8(w)) if wkind == "q8" else ("f32", shape, w)
    for k, n in (("qkv_b", 3 * width), ("proj_b", width), ("fc1_b", mlp), ("fc2_b", width)):
        p[k] = ("f32", (n,), r(n, std=0.02))
    for k in ("ln1", "ln2"):
        p[k + "_w"] = ("f32", (width,), r(width, std=0.1, mean=1.0))
        p[k + "_b"] = ("f32", (width,), r(width, std=0.1))
    return p


def _conv_plan(dim, d):
    """The neck's scales as lists of (op, output channels, kernel, GELU)."""
    head = [("conv", d, 1, False), ("conv", d, 3, False)]
    return [[("convT", dim // 2, 2, True), ("convT", dim // 4, 2, False)] + head,
            [("convT", dim // 2, 2, False)] + head, list(head), [("pool", 0, 2, False)] + head]


def _neck_params(r, dim, d):
    """(weight OHWI, bias) per convolution, scale by scale."""
    scales = []
    for plan in _conv_plan(dim, d):
        c, ws = dim, []
        for op, oc, k, _ in plan:
            if op == "pool":
                ws.append(None)
                continue
            ws.append((r(oc, k, k, c, std=0.02), r(oc, std=0.02)))
            c = oc
        scales.append(ws)
    return scales


def _inputs(case, seed):
    """The case's inputs on the GPU, by name."""
    r = _Rand(seed)
    kind = case["kind"]
    if kind == "text":
        return {"x": r(case["seq"], case["width"]),
                "p": [_layer_params(r, case["width"], "q8") for _ in range(case["layers"])]}
    if kind == "vit":
        return {"x": r(case["grid"] ** 2, case["width"]),
                "p": [_layer_params(r, case["width"], case["weights"])]}
    if kind == "neck":
        return {"x": r(1, case["grid"], case["grid"], case["dim"]),
                "p": _neck_params(r, case["dim"], case["d"])}
    if kind == "linear":
        t = TT[case["dtype"]]
        m, n, k = case["m"], case["n"], case["k"]
        return {"a": r(m, k).to(t), "w": r(*((n, k) if case["nt"] else (k, n)), std=0.02).to(t),
                "bias": r(n, std=0.01).to(t)}
    if kind == "q8":
        return {"a": r(case["m"], case["k"]).to(TT[case["a"]]),
                "w": _q8(r(case["n"], case["k"], std=0.02))}
    if kind == "q8batch":
        return {"a": r(case["m"], case["k"]),
                "w": _q8(r(case["copies"] * case["n"], case["k"], std=0.02))}
    if kind == "sdpa":
        t = TT[case["dtype"]]
        shape_q, shape_k = (case["bh"], case["sq"], HEAD), (case["bh"], case["sk"], HEAD)
        return {"q": r(*shape_q).to(t), "k": r(*shape_k).to(t), "v": r(*shape_k).to(t),
                "mask": r(case["sq"], case["sk"]) if case["mask"] else None}
    bh, s = case["bh"], case["s"]
    q, k, v = (r(bh, s, HEAD, std=0.125).to(torch.bfloat16) for _ in range(3))
    p = torch.empty(bh, s, s, dtype=torch.bfloat16, device=DEV)
    for i in range(0, bh, 64):  # probabilities: rows of a softmax
        p[i:i + 64] = torch.softmax(r(min(64, bh - i), s, s), -1).to(torch.bfloat16)
    return {"q": q, "k": k, "v": v, "p": p}


# ------------------------------------------------------------------ state
class _GraphState:
    """A backend with its weights mapped into HBM, and one graph whose input
    and outputs are device buffers."""

    def __init__(self):
        self.be = hip.Backend(0)
        self.G = graph.Graph()
        self.keep, self.parts, self.at, self.outs = [], [], 0, []

    def stage(self, kind, shape, t):
        """Take a tensor into the weight blob; its header comes with map()."""
        raw = t.contiguous().view(torch.uint8).reshape(-1)
        at = self.at
        self.parts.append((at, raw))
        self.at = (at + raw.numel() + 63) // 64 * 64  # a weight file's alignment
        return kind, list(shape), at, raw.numel()

    def map(self):
        """The blob to the host, as a weight file's mapping, and into HBM."""
        dev = torch.zeros(max(self.at, 64), dtype=torch.uint8, device=DEV)
        for at, raw in self.parts:
            dev[at:at + raw.numel()] = raw
        self.parts = []
        self.blob = dev.cpu().numpy()
        hip.check(self.be.map_weights(self.blob.ctypes.data, self.blob.nbytes), "map_weights")

    def weight(self, staged):
        kind, shape, at, nbytes = staged
        t = abi.make_tensor(abi.Q8_0 if kind == "q8" else abi.F32, shape,
                            self.blob.ctypes.data + at, nbytes)
        self.keep.append(t)
        return t

    def device(self, x, shape=None):
        t = abi.make_tensor(abi.F32, list(shape or x.shape), x.data_ptr(), x.numel() * 4)
        self.keep += [x, t]
        return t

    def output(self, t):
        """Put a graph output into a device buffer."""
        y = torch.empty(list(t.dims)[:t.n_dims], dtype=torch.float32, device=DEV)
        t.data = y.data_ptr()
        self.outs.append(y)

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.be.close()
        except Exception:
            pass


def _prepare_encoder(case, inp):
    s = _GraphState()
    staged = [{k: s.stage(*v) for k, v in p.items()} for p in inp["p"]]
    if case["kind"] == "vit":
        side = case["grid"] if case["global"] else case["window"]
        tabs = [s.stage("f32", t.shape, torch.from_numpy(t).to(DEV))
                for t in graph.rope_tables(side, HEAD)]
    else:
        m = torch.from_numpy(graph.causal_mask(case["seq"])).to(DEV)
        tabs = [s.stage("f32", m.shape, m)]
    s.map()
    tabs = [s.weight(t) for t in tabs]
    x = s.device(inp["x"])
    heads = case["width"] // HEAD
    for p in staged:
        p = {k: s.weight(v) for k, v in p.items()}
        x = (graph.vit_block(s.G, x, p, heads, case["grid"], case["window"], case["global"], *tabs)
             if case["kind"] == "vit" else graph.text_layer(s.G, x, p, heads, tabs[0]))
    s.output(x)
    s.G.g.no_readback = True
    return s


def _prepare_neck(case, inp):
    s = _GraphState()
    staged = [[w and (s.stage("f32", w[0].shape, w[0]), s.stage("f32", w[1].shape, w[1]))
               for w in ws] for ws in inp["p"]]
    s.map()
    G, x0, outs = s.G, s.device(inp["x"]), []
    for plan, ws in zip(_conv_plan(case["dim"], case["d"]), staged):
        t = x0
        for (op, oc, k, gelu), w in zip(plan, ws):
            _, h, wd, c = list(t.dims)
            if op == "pool":
                t = G.node(abi.OP_MAXPOOL2D, [t], G.tensor(abi.F32, (1, h // 2, wd // 2, c)),
                           (2, 2, 0, 0))
                continue
            wt, b = s.weight(w[0]), s.weight(w[1])
            if op == "convT":
                t = G.node(abi.OP_CONV_TRANSPOSE2D, [t, wt],
                           G.tensor(abi.F32, (1, 2 * h, 2 * wd, oc)), (2, 0, 0, 0))
            else:
                t = G.node(abi.OP_CONV2D, [t, wt], G.tensor(abi.F32, (1, h, wd, oc)),
                           (1, k // 2, 1, 0))
            t = G.node(abi.OP_BIAS_ADD, [t, b], G.tensor(abi.F32, list(t.dims)))
            if gelu:
                t = G.node(abi.OP_GELU, [t], G.tensor(abi.F32, list(t.dims)))
        outs.append(t)
    for t in outs:
        s.output(t)
    G.g.no_readback = True
    return s


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("text", "vit", "neck"):
        s = (_prepare_neck if kind == "neck" else _prepare_encoder)(case, inp)
        torch.cuda.synchronize()  # the backend works on a stream of its own
        return {"case": case, "graph": s}
    st = dict(inp, case=case)
    new = lambda *shape, t="f32": torch.empty(shape, dtype=TT[t], device=DEV)  # noqa: E731
    if kind == "linear":
        st["c"] = new(case["m"], case["n"], t=case["dtype"])
    elif kind == "q8":
        st["c"] = new(case["m"], case["n"])
    elif kind == "q8batch":
        st["c"] = new(case["copies"], case["m"], case["n"])
    elif kind == "sdpa":
        st["c"] = torch.empty_like(inp["q"])
    else:
        st["scores"] = new(case["bh"], case["s"], case["s"], t="bf16")
        st["c"] = new(case["bh"], case["s"], HEAD, t="bf16")
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("text", "vit", "neck"):
        s = state["graph"]
        hip.check(s.be.graph_eval(s.G.g), "graph_eval")
        return list(s.outs)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if kind == "linear":
        dt = DT[case["dtype"]]
        flags = ((hip.BIAS if case["bias"] else 0) | (hip.GELU if case["gelu"] else 0) |
                 (hip.B_NT if case["nt"] else 0))
        hip.matmul_dev(dt, state["a"].data_ptr(), dt, state["w"].data_ptr(), dt,
                       state["c"].data_ptr(), case["m"], case["n"], case["k"],
                       state["bias"].data_ptr() if case["bias"] else None, flags, stream)
        return state["c"]
    if kind == "q8":
        hip.matmul_dev(DT[case["a"]], state["a"].data_ptr(), abi.Q8_0, state["w"].data_ptr(),
                       abi.F32, state["c"].data_ptr(), case["m"], case["n"], case["k"], None,
                       hip.B_NT, stream)
        return state["c"]
    if kind == "q8batch":
        m, n, k = case["m"], case["n"], case["k"]
        hip.q8_batched_dev(abi.F32, state["a"].data_ptr(), state["w"].data_ptr(),
                           state["c"].data_ptr(), case["copies"], m, n, k, 0, n * k // 32 * 36,
                           m * n, None, 0, stream)
        return state["c"]
    lib = hip.load()
    if kind == "sdpa":
        mask = state["mask"].data_ptr() if case["mask"] else None
        hip.check(lib.sam3_hip_sdpa(DT[case["dtype"]], state["q"].data_ptr(), state["k"].data_ptr(),
                                    state["v"].data_ptr(), mask, state["c"].data_ptr(), case["bh"],
                                    case["sq"], case["sk"], HEAD, stream), "sdpa")
        return state["c"]
    bh, n = case["bh"], case["s"]
    hip.check(lib.sam3_hip_matmul_batched(abi.BF16, state["q"].data_ptr(), state["k"].data_ptr(),
                                          state["scores"].data_ptr(), bh, n, n, HEAD, n * HEAD,
                                          n * HEAD, n * n, hip.B_NT, stream), "scores")
    hip.check(lib.sam3_hip_matmul_batched(abi.BF16, state["p"].data_ptr(), state["v"].data_ptr(),
                                          state["c"].data_ptr(), bh, n, HEAD, n, n * n, n * HEAD,
                                          n * HEAD, 0, stream), "values")
    return [state["scores"], state["c"]]


# ------------------------------------------------------------------ the oracle
def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _ln(x, w, b):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt(d.square().mean(-1, keepdim=True) + 1e-5) * w + b


def _attend(q, k, v, mask=None):
    """softmax(q k^T / sqrt(D) + mask) v of [BH, S, D], a few heads at a time."""
    out = torch.empty_like(q)
    step = max(1, (1 << 27) // (q.shape[1] * k.shape[1]))
    for i in range(0, q.shape[0], step):
        s = torch.matmul(q[i:i + step], k[i:i + step].transpose(1, 2).contiguous())
        s = s / math.sqrt(q.shape[2]) + (mask if mask is not None else 0)
        out[i:i + step] = torch.matmul(torch.softmax(s, -1), v[i:i + step].contiguous())
    return out


def _rope(x, cos, sin):
    """Pairs (2i, 2i+1) of x [B, S, H, D] turned by the tables [S, D/2]."""
    a, b = x[..., 0::2], x[..., 1::2]
    c, s = cos[None, :, None, :], sin[None, :, None, :]
    return torch.stack((a * c - b * s, a * s + b * c), -1).reshape(x.shape)


def _exact_encoder(case, inp):
    x = inp["x"].double()
    width, n = case["width"], case["seq"] if case["kind"] == "text" else case["grid"] ** 2
    heads = width // HEAD
    windowed = case["kind"] == "vit" and not case["global"]
    ws = case["window"] if windowed else 0
    nw = case["grid"] // ws if windowed else 0
    for raw in inp["p"]:
        p = {k: _deq64(t, shape) if kind == "q8" else t.double()
             for k, (kind, shape, t) in raw.items()}
        y = _ln(x, p["ln1_w"], p["ln1_b"])
        if windowed:
            y = y.reshape(nw, ws, nw, ws * width).permute(0, 2, 1, 3).reshape(n, width)
        S = ws * ws if windowed else n
        qkv = (y @ p["qkv_w"].T + p["qkv_b"]).reshape(n // S, S, 3, heads, HEAD)
        q, k, v = (qkv[:, :, i] for i in range(3))
        mask = None
        if case["kind"] == "vit":
            cos, sin = (torch.from_numpy(t).to(DEV).double()
                        for t in graph.rope_tables(ws if windowed else case["grid"], HEAD))
            q, k = _rope(q, cos, sin), _rope(k, cos, sin)
        else:
            mask = torch.from_numpy(graph.causal_mask(n)).to(DEV).double()
        q, k, v = (t.permute(0, 2, 1, 3).reshape(-1, S, HEAD).contiguous() for t in (q, k, v))
        a = _attend(q, k, v, mask).reshape(n // S, heads, S, HEAD).permute(0, 2, 1, 3)
        a = a.reshape(n, width) @ p["proj_w"].T + p["proj_b"]
        if windowed:
            a = a.reshape(nw, nw, ws, ws * width).permute(0, 2, 1, 3).reshape(n, width)
        x = x + a
        y = _ln(x, p["ln2_w"], p["ln2_b"])
        x = x + (_gelu(y @ p["fc1_w"].T + p["fc1_b"]) @ p["fc2_w"].T + p["fc2_b"])
    return [x]


def _exact_neck(case, inp):
    outs = []
    for plan, ws in zip(_conv_plan(case["dim"], case["d"]), inp["p"]):
        x = inp["x"][0].double()
        for (op, oc, k, gelu), w in zip(plan, ws):
            h, wd, c = x.shape
            if op == "pool":
                x = x[:h // 2 * 2, :wd // 2 * 2].reshape(h // 2, 2, wd // 2, 2, c).amax((1, 3))
                continue
            wt, b = w[0].double(), w[1].double()
            if op == "convT":
                y = torch.empty(2 * h, 2 * wd, oc, dtype=torch.float64, device=DEV)
                for i in range(2):
                    for j in range(2):
                        y[i::2, j::2] = x @ wt[:, i, j].T
            else:
                pad = torch.zeros(h + k - 1, wd + k - 1, c, dtype=torch.float64, device=DEV)
                pad[k // 2:k // 2 + h, k // 2:k // 2 + wd] = x
                y = sum(pad[i:i + h, j:j + wd] @ wt[:, i, j].T for i in range(k) for j in range(k))
            x = y + b
            if gelu:
                x = _gelu(x)
        outs.append(x[None])
    return outs


def exact(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("text", "vit"):
        return _exact_encoder(case, inp)
    if kind == "neck":
        return _exact_neck(case, inp)
    if kind == "linear":
        w = inp["w"].double()
        y = inp["a"].double() @ (w.T if case["nt"] else w)
        if case["bias"]:
            y = y + inp["bias"].double()
        return _gelu(y) if case["gelu"] else y
    if kind == "q8":
        return inp["a"].double() @ _deq64(inp["w"], (case["n"], case["k"])).T
    if kind == "q8batch":
        w = _deq64(inp["w"], (case["copies"], case["n"], case["k"]))
        return torch.stack([inp["a"].double() @ x.T for x in w])
    if kind == "sdpa":
        mask = inp["mask"].double() if case["mask"] else None
        return _attend(inp["q"].double(), inp["k"].double(), inp["v"].double(), mask)
    q, k, v, p = (inp[t].double() for t in "qkvp")
    return [torch.matmul(q, k.transpose(1, 2).contiguous()), torch.matmul(p, v)]


# ------------------------------------------------------------------ accounts
def work(case):
    """Bytes (each input read once, each output written once) and flops."""
    kind = case["kind"]
    if kind in ("text", "vit"):
        e = case["width"]
        n = case["seq"] if kind == "text" else case["grid"] ** 2
        layers = case.get("layers", 1)
        S = n if kind == "text" or case["global"] else case["window"] ** 2
        wb = 36 / 32 if kind == "text" or case["weights"] == "q8" else 4
        return {"bytes": layers * (12 * e * e * wb + 13 * e * 4) + 2 * n * e * 4,
                "flops": layers * (24.0 * n * e * e + 4.0 * n * S * e)}
    if kind == "neck":
        flops, nbytes = 0.0, case["grid"] ** 2 * case["dim"] * 4
        for plan in _conv_plan(case["dim"], case["d"]):
            h, c = case["grid"], case["dim"]
            for op, oc, k, _ in plan:
                if op == "pool":
                    h //= 2
                    continue
                flops += 2.0 * h * h * c * oc * k * k
                nbytes += (oc * k * k * c + oc) * 4
                h, c = (2 * h, oc) if op == "convT" else (h, oc)
            nbytes += h * h * c * 4
        return {"bytes": nbytes, "flops": flops}
    if kind in ("linear", "q8", "q8batch"):
        m, n, k, b = case["m"], case["n"], case["k"], case.get("copies", 1)
        if kind == "linear":
            nbytes = 2 * (m * k + n * k + m * n + (n if case["bias"] else 0))
        else:
            nbytes = m * k * (2 if case.get("a") == "bf16" else 4) + b * (n * k / 32 * 36 + m * n * 4)
        return {"bytes": nbytes, "flops": 2.0 * b * m * n * k}
    if kind == "sdpa":
        es = 4 if case["dtype"] == "f32" else 2
        nbytes = case["bh"] * HEAD * es * 2 * (case["sq"] + case["sk"])
        return {"bytes": nbytes + (case["sq"] * case["sk"] * 4 if case["mask"] else 0),
                "flops": 4.0 * case["bh"] * case["sq"] * case["sk"] * HEAD}
    bh, s = case["bh"], case["s"]
    return {"bytes": bh * (2.0 * s * s * 2 + 4 * s * HEAD * 2), "flops": 4.0 * bh * s * s * HEAD}


def tolerance(case):
    """About four times what the paths show against float64 (measured over
    the listed and some drawn cases)."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 8e-3, "max": 0.05} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 8e-3}
    if kind == "attn":
        return {"rel": 7e-3, "max": 0.02}
    if kind == "sdpa":
        return {"f32": {"rel": 3e-5, "max": 4e-4}, "f16": {"rel": 1.5e-3, "max": 0.012},
                "bf16": {"rel": 1e-2, "max": 0.08}}[case["dtype"]]
    if kind == "neck":
        return {"rel": 4e-5, "max": 3e-4}
    if kind == "vit" and case["weights"] == "f32":
        return {"rel": 1.5e-5, "max": 1e-4}
    if kind == "text" and case["seq"] == 1:  # one token's products are f32
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 1.2e-3, "max": 8e-3}  # f16 operands against Q8_0 weights
