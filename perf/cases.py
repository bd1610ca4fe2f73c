"""What this library is asked to do in use, as cases that can be timed and compared.

A case is one pass of a Qwen3-MoE engine through the public entry points: a walk of the MoE
layers at one decode position (``layers``), the MoE half of the layer loop on a resident residual
stream (``chain``), the drop-in call on host buffers (``host``), the trunk's q/k/v and output
products of every layer (``trunk``), or the output head (``head``). Weights are seeded normals
packed into the GGUF block formats and resident in HBM once per model, as an engine keeps them; a
seed makes the activations. Layers differ in their weights and every state in its tokens, so a
decode pass does not find its experts in the memory-side cache.

The library promises the reference engine's bits, whatever the order a kernel works in, so the
results are compared exactly."""
import functools
import math

import numpy as np
import torch

from large_model_amd import qmsg
from large_model_amd.workloads import zipf_bias

TYPES = {"f32": qmsg.QMSG_T_F32, "f16": qmsg.QMSG_T_F16, "q4_0": qmsg.QMSG_T_Q4_0, "q4_1": qmsg.QMSG_T_Q4_1,
         "q8_0": qmsg.QMSG_T_Q8_0, "q6_k": qmsg.QMSG_T_Q6_K}
SHAPES = {  # n_embd, n_expert, n_used, n_ff_exp
    "tiny": (256, 16, 4, 128),          # random-init smoke-sized layer
    "small": (1024, 60, 4, 704),        # generic: an expert count that is no power of two
    "q30b": (2048, 128, 8, 768),        # Qwen3-30B-A3B
    "q235b": (4096, 128, 8, 1536),      # Qwen3-235B-A22B
}
TRUNKS = {  # n_embd, rows of q, rows of k and of v
    "small": (1024, 1536, 224),
    "q30b": (2048, 4096, 512),
    "q235b": (4096, 8192, 512),
}
MAX_TOKENS = 512
SIGMA = 0.02


def listed():
    return [
        # the smallest call: launches and latency only
        {"name": "tiny_t3", "op": "layers", "shape": "tiny", "gate": "q4_0", "down": "q4_0", "layers": 1, "T": 3, "zipf": False},
        # the call an engine that keeps its activations on the host makes (the reference's own call site)
        {"name": "q30b_host_t1", "op": "host", "shape": "q30b", "gate": "q4_0", "down": "q4_0", "layers": 4, "T": 1, "zipf": False},
        # batch-1 decode of the large model, Q4_0
        {"name": "q235b_decode_t1", "op": "layers", "shape": "q235b", "gate": "q4_0", "down": "q4_0", "layers": 4, "T": 1, "zipf": False},
        # a few sequences decoded together; Q4_1 down as the Q4_0 files hold it in some layers
        {"name": "q235b_decode_t5", "op": "layers", "shape": "q235b", "gate": "q4_0", "down": "q4_1", "layers": 2, "T": 5, "zipf": False},
        # a serving batch through the layer loop, Q6_K down
        {"name": "q235b_chain_t64", "op": "chain", "shape": "q235b", "gate": "q4_0", "down": "q6_k", "layers": 4, "T": 64, "zipf": False},
        # prefill with a skewed expert load
        {"name": "q235b_prefill_t512", "op": "layers", "shape": "q235b", "gate": "q4_0", "down": "q4_0", "layers": 1, "T": 512, "zipf": True},
        # a Q8_0 file: decode and an odd-sized prompt
        {"name": "q30b_q8_decode_t1", "op": "layers", "shape": "q30b", "gate": "q8_0", "down": "q8_0", "layers": 4, "T": 1, "zipf": False},
        {"name": "q30b_q8_prefill_t201", "op": "layers", "shape": "q30b", "gate": "q8_0", "down": "q8_0", "layers": 1, "T": 201, "zipf": True},
        # the trunk's products: decode, a ragged batch on the other block formats, prefill
        {"name": "trunk_decode_t1", "op": "trunk", "shape": "q235b", "q": "q4_0", "v": "q4_0", "o": "q4_0", "layers": 8, "T": 1},
        {"name": "trunk_mixed_t19", "op": "trunk", "shape": "q30b", "q": "q4_1", "v": "q6_k", "o": "q6_k", "layers": 4, "T": 19},
        {"name": "trunk_prefill_t512", "op": "trunk", "shape": "q235b", "q": "q4_0", "v": "q4_0", "o": "q4_0", "layers": 1, "T": 512},
        # output.weight at one position
        {"name": "head_t1", "op": "head", "cols": 4096, "rows": 151936, "q": "q6_k", "T": 1},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["layers", "layers", "layers", "chain", "host", "trunk", "trunk", "head"])
    T = _log_int(rng, 1, MAX_TOKENS)
    if op == "trunk":
        shape = rng.choice(["small", "q30b", "q235b"])
        # k and q share a type, as the files hold them; now and then v and o are wider
        quant = ["q4_0", "q4_0", "q4_1"] + (["q6_k"] if shape != "small" else [])
        q = rng.choice(quant + ["q8_0", "f32"])
        v, o = (q, q) if q in ("q8_0", "f32") else (rng.choice(quant), rng.choice(quant))
        if q in ("q8_0", "f32"):
            T = min(T, 256)
        return {"op": op, "shape": shape, "q": q, "v": v, "o": o, "layers": 1 if T > 16 else 4, "T": T}
    if op == "head":
        return {"op": op, "cols": rng.choice([2048, 4096]), "rows": rng.choice([32003, 100001, 151936]),
                "q": rng.choice(["q4_0", "q6_k", "q6_k"]), "T": _log_int(rng, 1, 8)}
    shape = rng.choice(["tiny", "small", "q30b", "q235b"])
    gate = rng.choice(["q4_0", "q4_0", "q4_0", "q4_1", "q6_k"] + (["q8_0", "f16"] if shape in ("small", "q30b") else []))
    if gate in ("q8_0", "f16"):
        down, T = gate, min(T, 201)
    else:
        down = rng.choice(["q4_0", "q4_0", "q4_1"] + (["q6_k"] if shape in ("q30b", "q235b") else []))
    layers = 1 if shape == "tiny" else (2 if T > 4 or shape == "q235b" else 4)
    if T > 64 or gate != "q4_0":
        layers = 1
    return {"op": op, "shape": shape, "gate": gate, "down": down, "layers": layers, "T": T, "zipf": T >= 64 and rng.random() < 0.5}


# ---- GGUF block formats ----

def _f16_bytes(d):
    return d.to(torch.float16).contiguous().view(torch.uint8).reshape(*d.shape, 2)


def pack(kind, w):
    """Rows w [rows][cols] (float32) as the format's row bytes [rows][row_bytes]."""
    rows, cols = w.shape
    if kind in ("f32", "f16"):
        return w.to(torch.float32 if kind == "f32" else torch.float16).contiguous().view(torch.uint8).reshape(rows, -1)
    if kind == "q6_k":
        b = w.reshape(rows, cols // 256, 16, 16)
        s = b.abs().amax(-1) / 31
        d = (s.amax(-1) / 127).to(torch.float16)
        sc = (s / d.float().unsqueeze(-1)).round().clamp(1, 127)
        c = (b / (d.float()[..., None, None] * sc[..., None])).round().clamp(-32, 31).to(torch.int32) + 32
        c = c.reshape(rows, cols // 256, 2, 4, 32).to(torch.uint8)        # half, group of 32, element
        lo, hi = c & 15, c >> 4
        ql = lo[:, :, :, 0:2] | (lo[:, :, :, 2:4] << 4)
        qh = hi[:, :, :, 0] | (hi[:, :, :, 1] << 2) | (hi[:, :, :, 2] << 4) | (hi[:, :, :, 3] << 6)
        out = torch.cat([ql.reshape(rows, -1, 128), qh.reshape(rows, -1, 64), sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)], -1)
        return out.reshape(rows, -1)
    b = w.reshape(rows, cols // 32, 32)
    if kind == "q8_0":
        d = (b.abs().amax(-1) / 127).to(torch.float16)
        c = (b / d.float().unsqueeze(-1)).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_f16_bytes(d), c], -1).reshape(rows, -1)
    if kind == "q4_0":
        top = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True)).squeeze(-1)
        d = (top / -8).to(torch.float16)
        c = (b / d.float().unsqueeze(-1) + 8.5).floor().clamp(0, 15).to(torch.uint8)
        head = _f16_bytes(d)
    else:                                                                  # q4_1
        m = b.amin(-1)
        d = ((b.amax(-1) - m) / 15).to(torch.float16)
        c = ((b - m.unsqueeze(-1)) / d.float().unsqueeze(-1)).round().clamp(0, 15).to(torch.uint8)
        head = torch.cat([_f16_bytes(d), _f16_bytes(m)], -1)
    return torch.cat([head, c[..., :16] | (c[..., 16:] << 4)], -1).reshape(rows, -1)


def unpack(kind, raw, cols):
    """The weights that row bytes stand for, in float64."""
    rows = raw.shape[0]

    def half(x):
        return x.contiguous().view(torch.float16).double()

    if kind in ("f32", "f16"):
        return raw.contiguous().view(torch.float32 if kind == "f32" else torch.float16).double()
    if kind == "q6_k":
        b = raw.reshape(rows, cols // 256, 210)
        ql, qh = b[..., :128].reshape(rows, -1, 2, 2, 32), b[..., 128:192].reshape(rows, -1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 3)
        hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 3)
        c = (lo | (hi << 4)).double().reshape(rows, -1, 16, 16) - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        return (c * (sc * half(b[..., 208:210])).unsqueeze(-1)).reshape(rows, cols)
    if kind == "q8_0":
        b = raw.reshape(rows, cols // 32, 34)
        return (b[..., 2:].contiguous().view(torch.int8).double() * half(b[..., :2])).reshape(rows, cols)
    n = 2 if kind == "q4_0" else 4
    b = raw.reshape(rows, cols // 32, 16 + n)
    c = torch.cat([b[..., n:] & 15, b[..., n:] >> 4], -1).double()
    c = (c - 8) * half(b[..., :2]) if kind == "q4_0" else c * half(b[..., :2]) + half(b[..., 2:4])
    return c.reshape(rows, cols)


def rows_of(key, kind, rows, cols):
    """The row bytes of one matrix; `key` says which."""
    g = torch.Generator("cuda").manual_seed(int(key))
    return pack(kind, torch.randn(rows, cols, generator=g, device="cuda") * SIGMA)


def _expert_key(layer, tensor, e):
    return 1000003 * (layer + 1) + 10007 * (tensor + 1) + e


def _router(shape, layer, zipf):
    E, X, K, F = SHAPES[shape]
    g = torch.Generator("cuda").manual_seed(77 + layer)
    r = torch.randn(X, E, generator=g, device="cuda") * SIGMA
    if zipf:                        # a bias per expert in column 0, whose input is 1
        r[:, 0] = torch.from_numpy(zipf_bias(X, K, MAX_TOKENS, E))
    return r


# ---- what an engine keeps: resident models ----

@functools.lru_cache(maxsize=4)
def model(shape, gate, down, layers, zipf):
    E, X, K, F = SHAPES[shape]
    ctx = qmsg.Context(E, X, K, F, n_layer=layers, max_tokens=MAX_TOKENS)
    for l in range(layers):
        host = []
        for i, (kind, rows, cols) in enumerate(((gate, F, E), (gate, F, E), (down, E, F))):
            buf = np.empty((X, rows * qmsg.row_bytes(TYPES[kind], cols)), np.uint8)
            for e in range(X):
                torch.from_numpy(buf[e]).copy_(rows_of(_expert_key(l, i, e), kind, rows, cols).reshape(-1))
            host.append((TYPES[kind], buf))
        ctx.upload(l, _router(shape, l, zipf).cpu().numpy(), *host)
        ctx.layer_norm(l, (1 + 0.1 * np.sin(np.arange(E) + l)).astype(np.float32))
    return ctx


def _trunk_mats(case):
    """Per layer, the q, k, v matrices of one product and the output projection: (key, type, rows, cols)."""
    if case["op"] == "head":
        return [([(5, case["q"], case["rows"], case["cols"])],)]
    E, q, kv = TRUNKS[case["shape"]]
    return [([(100 * l + 11, case["q"], q, E), (100 * l + 12, case["q"], kv, E), (100 * l + 13, case["v"], kv, E)],
             [(100 * l + 14, case["o"], E, q)]) for l in range(case["layers"])]


@functools.lru_cache(maxsize=4)
def trunk(*fields):
    ctx = qmsg.Context(*SHAPES["tiny"], n_layer=1, max_tokens=1)
    ids = [[[ctx.mat_upload(TYPES[kind], rows_of(key, kind, rows, cols).cpu().numpy(), rows, cols)
             for key, kind, rows, cols in mats] for mats in calls] for calls in _trunk_mats(dict(fields))]
    return ctx, ids


def _trunk_key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "T")))


# ---- the passes ----

def _inputs(case, seed):
    """The activations of a pass: normals, normalised row by row like a layer's input."""
    g = torch.Generator("cuda").manual_seed(int(seed))
    T = case["T"]
    if case["op"] in ("trunk", "head"):
        return [[torch.randn(T, mats[0][3], generator=g, device="cuda") for mats in calls] for calls in _trunk_mats(case)]
    E = SHAPES[case["shape"]][0]
    if case["op"] == "chain":       # the residual stream: rows of differing size
        return torch.randn(T, E, generator=g, device="cuda") * (0.5 + torch.rand(T, 1, generator=g, device="cuda"))
    x = torch.randn(case["layers"], T, E, generator=g, device="cuda")
    x /= x.square().mean(-1, keepdim=True).sqrt()
    if case["zipf"]:
        x[..., 0] = 1.0
    return x


def prepare(case, seed):
    op, T = case["op"], case["T"]
    x = _inputs(case, seed)
    if op in ("trunk", "head"):
        ctx, ids = trunk(*_trunk_key(case))
        calls, outs = [], []
        for xs, layer_ids, layer_mats in zip(x, ids, _trunk_mats(case)):
            for xi, call_ids, mats in zip(xs, layer_ids, layer_mats):
                ys = [torch.empty(T, rows, device="cuda") for _, _, rows, _ in mats]
                calls.append((call_ids, xi.data_ptr(), T, [y.data_ptr() for y in ys]))
                outs.append(ys)
        state = {"op": op, "ctx": ctx, "calls": calls, "x": x, "out": outs}
    else:
        ctx = model(case["shape"], case["gate"], case["down"], case["layers"], case["zipf"])
        state = {"op": op, "ctx": ctx, "x": x}
        if op == "host":
            state["x"] = [np.array(v) for v in x.cpu().numpy()]
        elif op == "chain":
            state["out"] = torch.empty_like(x)
            state["call"] = (0, case["layers"], state["out"].data_ptr(), T, 1e-6)
            state["copy"] = (state["out"].data_ptr(), x.data_ptr(), x.numel() * 4)
        else:
            state["out"] = torch.empty_like(x)
            state["calls"] = [(l, x[l].data_ptr(), T, state["out"][l].data_ptr()) for l in range(case["layers"])]
    torch.cuda.synchronize()        # the library works on its context's own stream
    return state


def run(state):
    ctx, op = state["ctx"], state["op"]
    if op in ("trunk", "head"):
        for call in state["calls"]:
            ctx.matmul_n_device(*call)
        return state["out"]
    if op == "host":
        return [ctx.moe(l, x) for l, x in enumerate(state["x"])]
    if op == "chain":               # the step's embeddings, then the layer loop in place
        ctx.calibrate_copy(*state["copy"])
        ctx.moe_chain(*state["call"])
        return state["out"]
    for call in state["calls"]:
        ctx.moe_device(*call)
    return state["out"]


# ---- what a pass cannot do without ----

def work(case):
    T = case["T"]
    if case["op"] in ("trunk", "head"):
        b = f = 0
        for calls in _trunk_mats(case):
            for mats in calls:
                b += 4 * T * mats[0][3]
                for _, kind, rows, cols in mats:
                    b += rows * qmsg.row_bytes(TYPES[kind], cols) + 4 * T * rows
                    f += 2 * T * rows * cols
        return {"bytes": b, "flops": f}
    E, X, K, F = SHAPES[case["shape"]]
    expert = 2 * F * qmsg.row_bytes(TYPES[case["gate"]], E) + E * qmsg.row_bytes(TYPES[case["down"]], F)
    distinct = X * (1 - (1 - K / X) ** T)                 # experts that T independent tokens reach
    return {"bytes": case["layers"] * (4 * X * E + distinct * expert + 8 * T * E),
            "flops": case["layers"] * (2 * T * X * E + 6 * T * K * E * F)}


def tolerance(case):
    return "exact"


# ---- the same in float64 ----

FAST = ("f32", "q4_0", "q4_1", "q6_k")


def _int8(x):
    """The activations that the quantised products see: 32-blocks rounded to 127 steps."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    return torch.where(d > 0, (b / torch.where(d > 0, d, 1.0)).round() * d, torch.zeros_like(b)).reshape(x.shape)


def _product(kind, raw, x, int8):
    return (_int8(x) if int8 and kind != "f32" else x) @ unpack(kind, raw, x.shape[-1]).T


def _moe(case, l, x):
    E, X, K, F = SHAPES[case["shape"]]
    int8 = case["gate"] in FAST
    p = torch.softmax(x @ _router(case["shape"], l, case["zipf"]).double().T, -1)
    wt, sel = p.topk(K, -1)
    wt = wt / wt.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(X):
        t, k = (sel == e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        g, u = (_product(case["gate"], rows_of(_expert_key(l, i, e), case["gate"], F, E), x[t], int8) for i in (0, 1))
        a = g / (1 + torch.exp(-g)) * u
        y = _product(case["down"], rows_of(_expert_key(l, 2, e), case["down"], E, F), a, int8)
        out.index_add_(0, t, wt[t, k].unsqueeze(-1) * y)
    return out


def exact(case, seed):
    x = _inputs(case, seed)
    if case["op"] in ("trunk", "head"):
        out = []
        for xs, calls in zip(x, _trunk_mats(case)):
            for xi, mats in zip(xs, calls):
                int8 = all(kind in FAST for _, kind, _, _ in mats)
                out.append([_product(kind, rows_of(key, kind, rows, cols), xi.double(), int8) for key, kind, rows, cols in mats])
        return out
    if case["op"] == "chain":
        h = x.double()
        E = h.shape[-1]
        for l in range(case["layers"]):
            w = torch.from_numpy((1 + 0.1 * np.sin(np.arange(E) + l)).astype(np.float32)).cuda().double()
            h = h + _moe(case, l, h / (h.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w)
        return h
    out = [_moe(case, l, x[l].double()) for l in range(case["layers"])]
    return [o.cpu().numpy() for o in out] if case["op"] == "host" else torch.stack(out)
