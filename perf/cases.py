"""The work a program gives this library, as cases that can be timed and checked.

The matrices are those of the 27B model whose geometry the loader checks (gguf_pq2.py): hidden
width 5120, FFN width 17408, attention width 6144, K/V width 1024, 248320 output tokens; a drawn
case also takes row shards of them.  Weights are PQ2_0 blocks with ternary codes (one code in a
thousand is 3) and fp16 scales |N(0, 0.02)| + 1e-4; activations are N(0, 1), which is what a
rotated activation looks like.  Kinds of case:

* prepass: RMSNorm, rotation and Q8_1 of the layer input of a prompt; for one token the rotation
  and Q8_1 alone;
* decode: the projections of consecutive layers for one token, captured once in a HIP graph
  and replayed, as a decode loop does;
* gemv: one projection of several layers for one token from a Q8_1 activation, in one graph;
* head: the output matrix for one token, from the residual row;
* batch: every projection of one layer for 2 to 16 sequences decoded together, in one graph;
* gemm: one projection for a prompt, or for as many sequences or draft tokens, called eagerly.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), os.pardir, "p40-kernel_amd"))
import bonsai_p40 as B  # noqa: E402

EMBD, FF, ATTN, KV, VOCAB = 5120, 17408, 6144, 1024, 248320
EPS = 1e-6
# (n_out, n_in) of every prompt projection: gate/up, down, linear-attention qkv, attention gate,
# attention output, full-attention q, k/v
SHAPES = [(FF, EMBD), (EMBD, FF), (10240, EMBD), (ATTN, EMBD), (EMBD, ATTN), (12288, EMBD), (KV, EMBD)]


def listed():
    return [
        # one row rotated and quantised between two host-side ops: the smallest call there is
        {"name": "prepass 1x5120", "kind": "prepass", "n": EMBD, "n_tok": 1},
        # the layer input of a long prompt
        {"name": "prepass 2048x5120", "kind": "prepass", "n": EMBD, "n_tok": 2048},
        # decode: three linear-attention layers and one full-attention layer, the model's period
        {"name": "decode 4 layers", "kind": "decode", "layers": 4, "first": 0},
        # the gate projection, layer after layer
        {"name": "gemv 17408x5120", "kind": "gemv", "n_out": FF, "n_in": EMBD, "count": 16},
        # the largest matrix of a decoded token
        {"name": "head 248320x5120", "kind": "head", "n_out": VOCAB},
        # a few sequences decoded together
        {"name": "batch 4", "kind": "batch", "n_tok": 4},
        {"name": "batch 12", "kind": "batch", "n_tok": 12},
        # a serving batch, or the draft tokens of several sequences
        {"name": "gemm 17408x5120x33", "kind": "gemm", "n_out": FF, "n_in": EMBD, "n_tok": 33, "ws": False},
        # a short prompt through the long-row projection
        {"name": "gemm 5120x17408x100", "kind": "gemm", "n_out": EMBD, "n_in": FF, "n_tok": 100, "ws": False},
        # a prompt of no round length
        {"name": "gemm 10240x5120x777", "kind": "gemm", "n_out": 10240, "n_in": EMBD, "n_tok": 777, "ws": False},
        # the usual prompt chunks, with the workspace that such a program keeps
        {"name": "gemm 17408x5120x512 ws", "kind": "gemm", "n_out": FF, "n_in": EMBD, "n_tok": 512, "ws": True},
        {"name": "gemm 17408x5120x2048 ws", "kind": "gemm", "n_out": FF, "n_in": EMBD, "n_tok": 2048, "ws": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shard(rng, n_out):
    """n_out whole, or one rank's rows of it, at times not a round number of them."""
    n = n_out // rng.choice([1, 1, 2, 4])
    return n - (rng.randrange(1, 64) if rng.random() < 0.25 else 0)


def draw(rng):
    kind = rng.choice(["prepass", "decode", "gemv", "batch", "gemm", "gemm", "gemm"])
    if kind == "prepass":
        return {"kind": kind, "n": rng.choice([EMBD, ATTN, FF]), "n_tok": _log_int(rng, 1, 2048)}
    if kind == "decode":
        return {"kind": kind, "layers": rng.randint(2, 4), "first": rng.randint(0, 3)}
    if kind == "gemv":
        n_out, n_in = rng.choice(SHAPES)
        return {"kind": kind, "n_out": _shard(rng, n_out), "n_in": n_in, "count": rng.randint(8, 16)}
    if kind == "batch":
        return {"kind": kind, "n_tok": rng.randint(2, 16)}
    n_out, n_in = rng.choice(SHAPES)
    return {"kind": kind, "n_out": _shard(rng, n_out), "n_in": n_in, "n_tok": _log_int(rng, 17, 2048),
            "ws": rng.random() < 0.5}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weights(n_out, n_in, g):
    """PQ2_0 rows of n_in columns."""
    blocks = n_out * (n_in // B.QK_PQ2)
    three = torch.tensor([sum((i // 3 ** k % 3) << (2 * k) for k in range(4)) for i in range(81)],
                         dtype=torch.uint8, device="cuda")
    codes = three[torch.randint(0, 81, (blocks * 32,), generator=g, device="cuda", dtype=torch.int32)]
    codes[torch.randint(0, codes.numel(), (max(1, codes.numel() // 250),), generator=g, device="cuda")] |= 3
    d = (torch.randn(blocks, generator=g, device="cuda").abs() * 0.02 + 1e-4).half()
    w = torch.empty((blocks, B.PQ2_BYTES), dtype=torch.uint8, device="cuda")
    w[:, :2] = d.view(torch.uint8).view(blocks, 2)
    w[:, 2:] = codes.view(blocks, 32)
    return w.view(-1)


# position j of a Q8_1 block holds element 16(j>>4) + 4(j&3) + ((j>>2)&3)
_ORDER = [16 * (j >> 4) + 4 * (j & 3) + ((j >> 2) & 3) for j in range(32)]


def _q8(x):
    """Token rows x as chunk-major Q8_1 bytes, with the Q8_1 values of every element (d * q)."""
    n_tok, n = x.shape
    c = x.view(n_tok, n // 32, 32)
    d = c.abs().amax(-1, keepdim=True) / 127
    q = torch.where(d > 0, c / torch.where(d > 0, d, torch.ones_like(d)), torch.zeros_like(c))
    q = torch.sign(q) * torch.floor(q.abs() + 0.5)
    q = q.clamp(-127, 127)
    d = d.half()
    out = torch.empty((n // 32, n_tok, B.Q81_BYTES), dtype=torch.uint8, device=x.device)
    out[:, :, :2] = d.view(torch.uint8).view(n_tok, n // 32, 2).transpose(0, 1)
    s = q.sum(-1).to(torch.int16).contiguous()
    out[:, :, 2:4] = s.view(torch.uint8).view(n_tok, n // 32, 2).transpose(0, 1)
    out[:, :, 4:] = q[:, :, _ORDER].to(torch.int8).view(torch.uint8).transpose(0, 1)
    return out.view(-1), (q.double() * d.double()).view(n_tok, n)


def _layer_shapes(index):
    """Attention projections that share the layer's input, and the attention output."""
    if index % 4 == 3:
        return [(12288, EMBD), (KV, EMBD), (KV, EMBD)], (EMBD, ATTN)
    return [(10240, EMBD), (ATTN, EMBD)], (EMBD, ATTN)


def _decode_inputs(case, g):
    layers = []
    for i in range(case["layers"]):
        first, out = _layer_shapes(case["first"] + i)
        L = {"first": first, "out": out}
        L["W"] = [_weights(*s, g) for s in first + [out, (FF, EMBD), (FF, EMBD), (EMBD, FF)]]
        L["x"], L["h"] = (torch.randn(EMBD, generator=g, device="cuda") for _ in range(2))
        L["attn"] = torch.randn(ATTN, generator=g, device="cuda")
        L["norm"] = [torch.randn(EMBD, generator=g, device="cuda") * 0.1 + 1 for _ in range(2)]
        layers.append(L)
    return layers


def _batch_inputs(case, g):
    first, out = _layer_shapes(0)
    shapes = first + [out, (FF, EMBD), (FF, EMBD), (EMBD, FF)]
    W = [_weights(*s, g) for s in shapes]
    x = [torch.randn((case["n_tok"], n), generator=g, device="cuda") for n in (EMBD, ATTN, EMBD, FF)]
    return shapes, W, x, [0] * len(first) + [1, 2, 2, 3]


def _captured(launches):
    """The launches as a graph, after one eager round."""
    launches()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launches()
    return graph


def _y(*shape):
    return torch.zeros(shape, dtype=torch.float32, device="cuda")


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "prepass":
        n, n_tok = case["n"], case["n_tok"]
        s = {"case": case, "x": torch.randn((n_tok, n), generator=g, device="cuda")}
        s["w"] = torch.randn(n, generator=g, device="cuda") * 0.1 + 1
        s["xq"] = torch.zeros(B.q8_bytes(n, n_tok), dtype=torch.uint8, device="cuda")
        return s
    if kind == "decode":
        layers = _decode_inputs(case, g)
        hq = torch.zeros(B.q8_bytes(FF), dtype=torch.uint8, device="cuda")
        ws = torch.zeros(B.ffn_workspace_bytes(FF), dtype=torch.uint8, device="cuda")
        ys = [[_y(n) for n, _ in L["first"]] + [_y(EMBD), _y(EMBD)] for L in layers]

        def launches():
            for L, y in zip(layers, ys):
                k = len(L["first"])
                B.rmsnorm_fwht_gemv_group(L["W"][:k], L["x"], L["norm"][0], None, y[:k],
                                          [n for n, _ in L["first"]], EMBD, EPS)
                B.fwht_gemv(L["W"][k], L["attn"], None, y[k], EMBD, ATTN)
                B.ffn_gate_up_swiglu(L["W"][k + 1], L["W"][k + 2], L["h"], L["norm"][1], None, None, hq, FF,
                                     EMBD, EPS, ws)
                B.gemv(L["W"][k + 3], hq, y[k + 1], EMBD, FF)

        return {"case": case, "keep": (layers, hq, ws), "graph": _captured(launches), "y": ys}
    if kind == "gemv":
        n_out, n_in = case["n_out"], case["n_in"]
        W = [_weights(n_out, n_in, g) for _ in range(case["count"])]
        xq = [_q8(torch.randn((1, n_in), generator=g, device="cuda"))[0] for _ in W]
        ys = [_y(n_out) for _ in W]

        def launches():
            for w, x, y in zip(W, xq, ys):
                B.gemv(w, x, y, n_out, n_in)

        return {"case": case, "keep": (W, xq), "graph": _captured(launches), "y": ys}
    if kind == "head":
        s = {"case": case, "W": _weights(case["n_out"], EMBD, g)}
        s["x"] = torch.randn(EMBD, generator=g, device="cuda")
        s["norm"] = torch.randn(EMBD, generator=g, device="cuda") * 0.1 + 1
        s["y"] = _y(case["n_out"])
        return s
    if kind == "batch":
        n_tok = case["n_tok"]
        shapes, W, x, which = _batch_inputs(case, g)
        xq = [_q8(t)[0] for t in x]
        ys = [_y(n, n_tok) for n, _ in shapes]

        def launches():
            for (n_out, n_in), w, k, y in zip(shapes, W, which, ys):
                B.gemm(w, xq[k], y, n_out, n_in, n_tok)

        return {"case": case, "keep": (W, xq), "graph": _captured(launches), "y": ys}
    n_out, n_in, n_tok = case["n_out"], case["n_in"], case["n_tok"]
    s = {"case": case, "W": _weights(n_out, n_in, g)}
    s["xq"] = _q8(torch.randn((n_tok, n_in), generator=g, device="cuda"))[0]
    s["y"] = _y(n_out, n_tok)
    if case["ws"]:
        s["ws"] = torch.zeros(max(16, B.gemm_workspace_bytes(n_in, n_tok)), dtype=torch.uint8, device="cuda")
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if "graph" in state:
        state["graph"].replay()
        return state["y"]
    if kind == "prepass":
        if case["n_tok"] == 1:
            B.fwht_quant(state["x"], None, state["xq"], case["n"])
        else:
            B.rmsnorm_fwht_quant(state["x"], state["w"], None, state["xq"], case["n"], case["n_tok"], EPS)
        return state["xq"]
    if kind == "head":
        B.rmsnorm_fwht_gemv_group([state["W"]], state["x"], state["norm"], None, [state["y"]], [case["n_out"]],
                                  EMBD, EPS)
        return state["y"]
    if case["ws"]:
        B.gemm_ws(state["W"], state["xq"], state["y"], case["n_out"], case["n_in"], case["n_tok"], state["ws"])
    else:
        B.gemm(state["W"], state["xq"], state["y"], case["n_out"], case["n_in"], case["n_tok"])
    return state["y"]


# ---------------------------------------------------------- work, exactness
def _work_shapes(case):
    """(n_out, n_in) of every matrix product of a case and its token count."""
    if case["kind"] == "decode":
        shapes = []
        for i in range(case["layers"]):
            first, out = _layer_shapes(case["first"] + i)
            shapes += first + [out, (FF, EMBD), (FF, EMBD), (EMBD, FF)]
        return shapes, 1
    if case["kind"] == "gemv":
        return [(case["n_out"], case["n_in"])] * case["count"], 1
    if case["kind"] == "head":
        return [(case["n_out"], EMBD)], 1
    if case["kind"] == "batch":
        first, out = _layer_shapes(0)
        return first + [out, (FF, EMBD), (FF, EMBD), (EMBD, FF)], case["n_tok"]
    return [(case["n_out"], case["n_in"])], case["n_tok"]


def work(case):
    if case["kind"] == "prepass":
        n, t = case["n"], case["n_tok"]
        return {"bytes": 4 * n * t + (4 * n if t > 1 else 0) + B.q8_bytes(n, t), "flops": 12 * n * t}
    shapes, t = _work_shapes(case)
    nbytes = sum(B.pq2_bytes(*s) + t * (B.q8_bytes(s[1]) + 4 * s[0]) for s in shapes)
    return {"bytes": nbytes, "flops": sum(2 * a * b * t for a, b in shapes)}


def tolerance(case):
    if case["kind"] == "prepass":
        return "exact"                # one documented order of operations: the bytes are the contract
    if case["kind"] in ("decode", "head"):
        # sums in another order move an activation at a rounding tie by one of its 255 steps, and each
        # such step is about 1 / (30 sqrt(n_in)) of the output
        return {"rel": 1e-3}
    return {"rel": 2e-6, "max": 2e-5}


def _plain(w, n_out, n_in):
    """PQ2_0 rows as float64."""
    b = w.view(n_out, n_in // B.QK_PQ2, B.PQ2_BYTES)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    c = torch.stack([(b[:, :, 2:] >> (2 * k)) & 3 for k in range(4)], -1).view(n_out, n_in // B.QK_PQ2, 128)
    return ((c.double() - 1) * d).view(n_out, n_in)


def _rotated_q8(x):
    """Q8_1 values of the rotated row, in 64 bits."""
    h = torch.ones((1, 1), dtype=torch.float64, device="cuda")
    for _ in range(10):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return _q8((x.double().view(-1, B.HBLK) @ h / 32).view(1, -1))[1][0]


def _normed(x, w):
    x = x.double()
    return x * torch.rsqrt((x * x).mean() + EPS) * w.double()


def _product(w, n_out, n_in, x):
    """The matrix times x^T, rows of it at a time."""
    rows = max(1, (1 << 27) // n_in)
    out = []
    for r in range(0, n_out, rows):
        m = min(rows, n_out - r)
        part = w[B.pq2_bytes(r, n_in):B.pq2_bytes(r + m, n_in)]
        out.append(_plain(part, m, n_in) @ x.t())
    return torch.cat(out)


def exact(case, seed):
    if case["kind"] == "prepass":
        return None                   # bytes: held to "exact"
    g = _generator(seed)
    kind = case["kind"]
    if kind == "decode":
        out = []
        for L in _decode_inputs(case, g):
            k = len(L["first"])
            W = L["W"]
            a = _rotated_q8(_normed(L["x"], L["norm"][0]))
            y = [_product(W[i], n, EMBD, a[None])[:, 0] for i, (n, _) in enumerate(L["first"])]
            y.append(_product(W[k], EMBD, ATTN, _rotated_q8(L["attn"])[None])[:, 0])
            a = _rotated_q8(_normed(L["h"], L["norm"][1]))
            gate, up = (_product(W[k + 1 + i], FF, EMBD, a[None])[:, 0] for i in range(2))
            h = gate / (1 + torch.exp(-gate)) * up
            y.append(_product(W[k + 3], EMBD, FF, _rotated_q8(h)[None])[:, 0])
            out.append(y)
        return out
    if kind == "gemv":
        n_out, n_in = case["n_out"], case["n_in"]
        W = [_weights(n_out, n_in, g) for _ in range(case["count"])]
        x = [_q8(torch.randn((1, n_in), generator=g, device="cuda"))[1] for _ in W]
        return [_product(w, n_out, n_in, v)[:, 0] for w, v in zip(W, x)]
    if kind == "head":
        w = _weights(case["n_out"], EMBD, g)
        x = torch.randn(EMBD, generator=g, device="cuda")
        norm = torch.randn(EMBD, generator=g, device="cuda") * 0.1 + 1
        return _product(w, case["n_out"], EMBD, _rotated_q8(_normed(x, norm))[None])[:, 0]
    if kind == "batch":
        shapes, W, x, which = _batch_inputs(case, g)
        v = [_q8(t)[1] for t in x]
        return [_product(w, n_out, n_in, v[k]) for (n_out, n_in), w, k in zip(shapes, W, which)]
    w = _weights(case["n_out"], case["n_in"], g)
    v = _q8(torch.randn((case["n_tok"], case["n_in"]), generator=g, device="cuda"))[1]
    return _product(w, case["n_out"], case["n_in"], v)
