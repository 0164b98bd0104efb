"""Measured workloads of the package: what a serving program has it do, through its public entry points.

A case is one pass of a program that holds quantised weights or a KV cache on the GPU:

* ``linear``  one eager call of the int8 linear op.
* ``decode``  the four linears (qkv, o_proj, gate_up, down) of several dense layers at a decode or verification width
  (M <= 16), captured once in a HIP graph and replayed, as a server replays its decode step.
* ``prefill`` the same linears of one layer above 16 rows, called eagerly, as servers run prefill chunks and larger
  batches: ``arith`` "w8a8" is the default route of the op, "w8a16" the QWEN_FAST_LINEAR_PREFILL=w8a16 one.
* ``draft``   one draft step of the int8 LM head: the token ids, or the logits.
* ``attn``    verification attention over a paged KV cache, replayed as a graph of several layers or called eagerly.
* ``load``    the load-time quantisation of an LM head into the int8 image the draft step reads.

Inputs: int8 weights uniform in [-127, 127] with per-channel fp32 scales |N(0,1)| * 0.002 + 1e-4, bf16 N(0,1)
activations, queries, keys and values, shuffled cache pages; everything from the seed alone.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "qwen-a100-fastpath_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qwen_fastpath as qf  # noqa: E402

DEV = "cuda:0"
GEMMS = ("qkv", "o_proj", "gate_up", "down")


def _layer(qkv, attn, hidden, ffn2, ffn):
    """Sizes of one layer's linears: qkv hidden -> qkv, o_proj attn -> hidden, gate_up hidden -> ffn2, down ffn -> hidden."""
    return {"qkv": qkv, "attn": attn, "hidden": hidden, "ffn2": ffn2, "ffn": ffn}


_DENSE = _layer(10240, 8192, 5120, 34816, 17408)  # the dense 27B-class layer of the benchmark


def listed():
    return [
        # the smallest call: one token through one linear, eager
        {"name": "linear_m1", "kind": "linear", "M": 1, "N": 5120, "K": 5120, "layout": "tiled", "bias": True},
        # the benchmark's verification step (1 verified + 4 draft tokens), weights in the default load-time image
        {"name": "decode_m5", "kind": "decode", "M": 5, "layers": 8, "layout": "tiled", **_DENSE},
        # the same layers kept in the checkpoint's layout (QWEN_FAST_LINEAR_LAYOUT=rowmajor), an odd batch width
        {"name": "decode_m11_rowmajor", "kind": "decode", "M": 11, "layers": 4, "layout": "rowmajor", **_DENSE},
        # one rank's share of the layer at tensor parallelism 8: every linear is short
        {"name": "decode_m5_tp8", "kind": "decode", "M": 5, "layers": 8, "layout": "tiled",
         **_layer(1280, 1024, 5120, 4352, 2176)},
        # one draft step of single-user decode over the 151936-token vocabulary, padded head
        {"name": "draft_m1", "kind": "draft", "M": 1, "V": 151936, "H": 5120, "pad": 267, "out": "ids", "layout": "tiled"},
        # a short chat's verification step: 16 full-attention layers, 1000 cached positions
        {"name": "attn_1k", "kind": "attn", "Q": 3, "B": 1, "ctx": 1000, "step": 0, "H": 24, "HKV": 4, "D": 256,
         "page": 800, "layers": 16, "graph": True},
        # a long document's: 38000 positions
        {"name": "attn_38k", "kind": "attn", "Q": 3, "B": 1, "ctx": 38000, "step": 0, "H": 24, "HKV": 4, "D": 256,
         "page": 800, "layers": 4, "graph": True},
        # several users with ragged contexts, small pages, a wider verification window, called eagerly
        {"name": "attn_batch", "kind": "attn", "Q": 5, "B": 6, "ctx": 9000, "step": 1333, "H": 32, "HKV": 4, "D": 128,
         "page": 16, "layers": 4, "graph": False},
        # a batch of 8 users x 5 verified tokens: above the decode width
        {"name": "batch_m40", "kind": "prefill", "M": 40, "arith": "w8a8", "layout": "tiled", **_DENSE},
        # a short prompt of odd length
        {"name": "prefill_m333", "kind": "prefill", "M": 333, "arith": "w8a8", "layout": "tiled", **_DENSE},
        # a full prefill chunk
        {"name": "prefill_m4096", "kind": "prefill", "M": 4096, "arith": "w8a8", "layout": "tiled", **_DENSE},
        # loading: the 151936 x 5120 head quantised and laid out
        {"name": "load_head", "kind": "load", "V": 151936, "H": 5120, "layout": "tiled"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "decode", "decode", "prefill", "prefill", "prefill", "draft", "attn", "attn", "load"])
    if kind == "linear":
        return {"kind": kind, "M": rng.randint(1, 16), "N": _log_int(rng, 512, 16384), "K": 64 * _log_int(rng, 8, 256),
                "layout": rng.choice(["tiled", "tiled", "rowmajor"]), "bias": rng.random() < 0.5}
    if kind in ("decode", "prefill"):
        hidden, attn, ffn = 64 * _log_int(rng, 16, 96), 64 * _log_int(rng, 16, 128), 64 * _log_int(rng, 32, 272)
        c = {"kind": kind, **_layer(8 * _log_int(rng, 128, 1280), attn, hidden, 2 * ffn, ffn),
             "layout": rng.choice(["tiled", "tiled", "rowmajor"])}
        if kind == "decode":
            c.update(M=rng.randint(1, 16), layers=4)
        else:
            c.update(arith="w8a8", M=_log_int(rng, 17, 4096))
            if c["layout"] == "tiled" and rng.random() < 0.25:
                c.update(arith="w8a16", M=_log_int(rng, 17, 1024))
        return c
    if kind == "draft":
        return {"kind": kind, "M": rng.randint(1, 8), "V": _log_int(rng, 16000, 152000), "H": 64 * rng.randint(32, 80),
                "pad": rng.randint(0, 300), "out": rng.choice(["ids", "ids", "logits"]),
                "layout": rng.choice(["tiled", "tiled", "rowmajor"])}
    if kind == "attn":
        G, Q, B = rng.choice([2, 4, 6, 7, 8]), rng.randint(2, 8), rng.randint(1, 8)
        ctx = _log_int(rng, 300, 60000 // B)
        HKV = rng.choice([2, 4, 8])
        return {"kind": kind, "Q": Q, "B": B, "ctx": ctx, "step": rng.randint(0, ctx // 10), "H": G * HKV, "HKV": HKV,
                "D": rng.choice([64, 128, 128, 256, 256]), "page": rng.choice([16, 64, 800]), "layers": 4,
                "graph": rng.random() < 0.5}
    return {"kind": kind, "V": _log_int(rng, 16000, 152000), "H": 64 * rng.randint(32, 80),
            "layout": rng.choice(["tiled", "tiled", "rowmajor"])}


# ---- inputs ----

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _weight(g, N, K):
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
    s = torch.randn(N, device=DEV, generator=g).abs() * 0.002 + 1e-4
    return w, s


def _bf16(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g).to(torch.bfloat16)


def _shapes(case):
    return {"qkv": (case["qkv"], case["hidden"]), "o_proj": (case["hidden"], case["attn"]),
            "gate_up": (case["ffn2"], case["hidden"]), "down": (case["hidden"], case["ffn"])}


def _stack(case, seed):
    """The layers' linears in order: (N, K, x [M, K], w [N, K], s [N]), one at a time."""
    g = _gen(seed)
    for _ in range(case.get("layers", 1)):
        for name in GEMMS:
            N, K = _shapes(case)[name]
            x = _bf16(g, case["M"], K)
            yield (N, K, x) + _weight(g, N, K)


def _linear(case, seed):
    g = _gen(seed)
    x = _bf16(g, case["M"], case["K"])
    w, s = _weight(g, case["N"], case["K"])
    return x, w, s, _bf16(g, case["N"]) if case["bias"] else None


def _head(case, seed):
    """Draft-head inputs: each hidden state leans towards one unpadded token, as a trained head's does."""
    g = _gen(seed)
    w, s = _weight(g, case["V"], case["H"])
    tok = torch.randint(0, case["V"] - case["pad"], (case["M"],), device=DEV, generator=g)
    s[tok] = s[tok].clamp_min(0.004)
    x = torch.randn(case["M"], case["H"], device=DEV, generator=g) + w[tok].float() * (0.5 / 73.0)
    return x.to(torch.bfloat16), w, s, tok


def _attn_inputs(case, seed):
    g = _gen(seed)
    Q, B, H, HKV, D, page = (case[k] for k in ("Q", "B", "H", "HKV", "D", "page"))
    lens = [max(case["ctx"] - b * case["step"], 1) + Q for b in range(B)]
    nblk = (max(lens) + page - 1) // page + 1
    pages = B * nblk + 5
    table = torch.randperm(pages, device=DEV, generator=g)[:B * nblk].reshape(B, nblk).to(torch.int32)
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    per_layer = [(_bf16(g, B * Q, H, D), _bf16(g, pages, HKV, page, 2 * D)) for _ in range(case["layers"])]
    return lens, table, seq, per_layer


def _capture(fn):
    """fn's outputs and the HIP graph that recomputes them in place."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def prepare(case, seed):
    kind = case["kind"]
    tiled = case.get("layout") == "tiled"
    if kind == "linear":
        x, w, s, bias = _linear(case, seed)
        w = qf.to_tiled(w.t()) if tiled else w.t()
        return {"kind": kind, "x": x, "w": w, "s": s, "bias": bias}
    if kind in ("decode", "prefill"):
        parts = []
        for N, K, x, w, s in _stack(case, seed):
            parts.append((x, qf.to_tiled(w.t()) if tiled else w.t(), s))
            del w
        if kind == "prefill":
            return {"kind": kind, "parts": parts, "arith": case["arith"]}

        def step():
            return [qf.qf_int8_linear(x, w, s, None) for x, w, s in parts]

        graph, out = _capture(step)
        return {"kind": kind, "parts": parts, "graph": graph, "out": out}
    if kind == "draft":
        x, w, s, _ = _head(case, seed)
        layout = qf.TILED if tiled else qf.ROWMAJOR
        V, H = w.shape
        head = qf.Int8Head(qf.to_tiled(w.t()) if tiled else w.t(), s, case["pad"], qf.pick_config(V, H, layout), layout)
        return {"kind": kind, "x": x, "head": head, "out": case["out"]}
    if kind == "attn":
        lens, table, seq, per_layer = _attn_inputs(case, seed)
        calls = []
        for q, kv in per_layer:
            k, v = kv.transpose(1, 2).split(case["D"], dim=-1)
            calls.append((q, k, v, torch.empty_like(q)))

        def step():
            for q, k, v, o in calls:
                qf.gqa_packed_spec_attention(q, k, v, o, seq, table, case["B"], case["Q"], case["HKV"], case["D"] ** -0.5)
            return [o for _, _, _, o in calls]

        if case["graph"]:
            graph, out = _capture(step)
            return {"kind": kind, "keep": (calls, seq, table), "graph": graph, "out": out}
        return {"kind": kind, "step": step}
    return {"kind": kind, "w": (_bf16(_gen(seed), case["V"], case["H"]).float() * 0.02).to(torch.bfloat16),
            "layout": qf.TILED if tiled else qf.ROWMAJOR}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return qf.qf_int8_linear(state["x"], state["w"], state["s"], state["bias"])
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if kind == "prefill":
        if state["arith"] == "w8a16":
            return [qf.w8a16_mm(x, w, s, None, torch.bfloat16, qf.TILED) for x, w, s in state["parts"]]
        return [qf.qf_int8_linear(x, w, s, None) for x, w, s in state["parts"]]
    if kind == "draft":
        if state["out"] == "ids":
            return qf.int8_top_tokens(state["head"], state["x"])
        return qf.int8_logits(state["head"], state["x"])
    if kind == "attn":
        return state["step"]()
    head = qf.make_int8_head(state["w"], 0, state["layout"])
    return head.w_t if head.layout == qf.TILED else head.w_t.t(), head.scale


# ---- what a pass cannot do without ----

def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K + 4 * N + 2 * M * K + 2 * M * N + (2 * N if case["bias"] else 0), "flops": 2 * M * N * K}
    if kind in ("decode", "prefill"):
        M, n = case["M"], case.get("layers", 1)
        shapes = _shapes(case).values()
        return {"bytes": n * sum(N * K + 4 * N + 2 * M * (N + K) for N, K in shapes),
                "flops": n * sum(2 * M * N * K for N, K in shapes)}
    if kind == "draft":
        M, V, H = case["M"], case["V"], case["H"]
        return {"bytes": V * H + 4 * V + 2 * M * H + (8 * M if case["out"] == "ids" else 2 * M * V), "flops": 2 * M * V * H}
    if kind == "attn":
        Q, B, H, HKV, D = (case[k] for k in ("Q", "B", "H", "HKV", "D"))
        pos = sum(max(case["ctx"] - b * case["step"], 1) + Q for b in range(B))
        n = case["layers"]
        return {"bytes": n * (pos * HKV * 2 * D * 2 + 2 * B * Q * H * D * 2 + 4 * pos // case["page"]),
                "flops": n * 4 * pos * Q * H * D}
    return {"bytes": case["V"] * (3 * case["H"] + 4), "flops": 0}


def tolerance(case):
    if case["kind"] == "load" or (case["kind"] == "draft" and case["out"] == "ids"):
        return "exact"
    if case["kind"] == "attn":
        # softmax weights and outputs rounded to bf16 (weights 2^-9 relative each): another order of the sums moves
        # roundings of both
        return {"rel": 8e-3, "max": 0.05}
    # W8A16: fp32 sums in another order flip the bf16 rounding of about 2 outputs in 10000, most of them small ones
    # (a 2048-channel product in two orders: rel 4e-9 to 3e-8); W8A8: exact integer sums, only the order of the two
    # fp32 scale products is free.  One flip (2^-8 of a value) among 512 outputs is 2e-4.
    return {"rel": 5e-4, "max": 0.016}


# ---- the same results in 64 bits ----

def _exact_linear(x, w, s):
    """(x @ w^T) * s in 64 bits, in blocks of output channels."""
    xd = x.double()
    return torch.cat([(xd @ w[n:n + 8192].double().t()) * s[n:n + 8192].double() for n in range(0, w.shape[0], 8192)], 1)


def _exact_w8a8(x, w, s):
    """The per-token int8 linear: fp32 scale amax * fl(1/127) and half-to-even rounding of x / scale define the int8
    activations; sums and scales in 64 bits."""
    xf = x.float()
    sa = xf.abs().amax(1, keepdim=True) * torch.tensor(1.0 / 127.0, dtype=torch.float32, device=x.device)
    xq = torch.where(sa > 0, torch.round(xf / torch.where(sa > 0, sa, torch.ones_like(sa))), torch.zeros_like(xf))
    return _exact_linear(xq.clamp(-128, 127), w, s) * sa.double()


def _exact_attn(case, seed):
    lens, table, _, per_layer = _attn_inputs(case, seed)
    Q, HKV, D = case["Q"], case["HKV"], case["D"]
    G = case["H"] // HKV
    outs = []
    for q, kv in per_layer:
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b, n in enumerate(lens):
            rows = kv[table[b].long()].transpose(1, 2).reshape(-1, HKV, 2 * D)[:n]
            seen = torch.arange(n, device=DEV)[None, :] <= n - Q + torch.arange(Q, device=DEV)[:, None]
            for h in range(HKV):
                k, v = rows[:, h, :D].double(), rows[:, h, D:].double()
                qh = q[b * Q:(b + 1) * Q, h * G:(h + 1) * G].double()
                sc = (qh.reshape(Q * G, D) @ k.t()).reshape(Q, G, n) * D ** -0.5
                p = torch.softmax(sc.masked_fill(~seen[:, None, :], float("-inf")), -1)
                out[b * Q:(b + 1) * Q, h * G:(h + 1) * G] = (p.reshape(Q * G, n) @ v).reshape(Q, G, D)
        outs.append(out)
    return outs


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, s, bias = _linear(case, seed)
        y = _exact_linear(x, w, s)
        return y if bias is None else y + bias.double()
    if kind == "decode" or (kind == "prefill" and case["arith"] == "w8a16"):
        return [_exact_linear(x, w, s) for _, _, x, w, s in _stack(case, seed)]
    if kind == "prefill":
        return [_exact_w8a8(x, w, s) for _, _, x, w, s in _stack(case, seed)]
    if kind == "draft":
        if case["out"] == "ids":
            return None
        x, w, s, _ = _head(case, seed)
        return _exact_linear(x, w, s)
    if kind == "attn":
        return _exact_attn(case, seed)
    w = (_bf16(_gen(seed), case["V"], case["H"]).float() * 0.02).to(torch.bfloat16)
    scale = w.abs().amax(1).double().clamp_min(1e-8) / 127
    return [None, scale]
