"""The work that a user of this library has it do, as timed and compared cases.

The shapes are the reference model's (hidden 2560, FFN 10240, 16 query and 4
kv heads of 256 elements, three sliding layers of 512 positions to one full
layer). A whole-model case runs one period of four layers and a ninth of the
vocabulary (four of 36 layers), so the head keeps its share of a pass; the
weights still exceed every cache.

What the listed cases stand for:

  matvec-kv       the smallest call: one key or value projection, one f32
                  column, as the reference's C-ABI callers issue it
  gate-up         the largest pair of a decode step, one bf16 column
  down-5-f32      a draft of five tokens verified at the reference's f32
  q6k-layer       one layer's matvecs of the Q6_K trunk, recorded as a plan
  head-8          the tied Q8_0 head over a verify block
  prefill-up      a full prompt chunk through one FFN matrix
  prefill-down-77 a short prompt through the other, f32, an odd token count
  decode-1k       one token early in a conversation
  decode-30k      one token late in a long one
  verify-8        a block of drafted tokens in a medium context
  prompt-185      a user's turn: a ragged chunk after a few cached positions
  prompt-512-16k  a full chunk deep in a long document
"""
import concurrent.futures
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "spark-x2.6-4b-q6k_amd"))
import sparkmv as sm  # noqa: E402

HIDDEN, FFN, HEADS, KV_HEADS, HEAD_DIM, WINDOW = 2560, 10240, 16, 4, 256, 512
QD, KVD = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
LAYERS, VOCAB, HEAD_ROWS = 4, 16384, 151936
ROPE = ((1.0e4, 1.0), (5.0e6, 0.25))     # theta and rotated share: sliding, full layers
EPS = 1.0e-6
LAYER_MATS = (("qkv", QD + 2 * KVD, HIDDEN), ("attn_gate", HEADS, HIDDEN), ("out", HIDDEN, QD),
              ("gate", FFN, HIDDEN), ("up", FFN, HIDDEN), ("down", HIDDEN, FFN))


def listed():
    return [
        {"name": "matvec-kv", "kind": "vq", "rows": KVD, "cols": HIDDEN, "mats": 1, "ncols": 1, "x": "f32"},
        {"name": "gate-up", "kind": "vq", "rows": FFN, "cols": HIDDEN, "mats": 2, "ncols": 1, "x": "bf16"},
        {"name": "down-5-f32", "kind": "vq", "rows": HIDDEN, "cols": FFN, "mats": 1, "ncols": 5, "x": "f32"},
        {"name": "q6k-layer", "kind": "q6k-layer", "ncols": 1, "x": "bf16"},
        {"name": "head-8", "kind": "q8_0", "rows": HEAD_ROWS, "cols": HIDDEN, "ncols": 8, "x": "bf16"},
        {"name": "prefill-up", "kind": "prefill", "rows": FFN, "cols": HIDDEN, "tokens": 512, "x": "bf16"},
        {"name": "prefill-down-77", "kind": "prefill", "rows": HIDDEN, "cols": FFN, "tokens": 77, "x": "f32"},
        {"name": "decode-1k", "kind": "decode", "tokens": 1, "pos": 1003, "max_ctx": 8192, "x": "bf16"},
        {"name": "decode-30k", "kind": "decode", "tokens": 1, "pos": 30007, "max_ctx": 32768, "x": "bf16"},
        {"name": "verify-8", "kind": "verify", "tokens": 8, "pos": 6001, "max_ctx": 8192, "x": "bf16"},
        {"name": "prompt-185", "kind": "prompt", "tokens": 185, "pos": 37, "max_ctx": 8192, "x": "bf16"},
        {"name": "prompt-512-16k", "kind": "prompt", "tokens": 512, "pos": 16384, "max_ctx": 32768, "x": "bf16"},
    ]


def _log(rng, lo, hi):
    """An integer in lo .. hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["vq", "q6_k", "q8_0", "prefill", "decode", "verify", "prompt", "prompt"])
    x = rng.choice(["bf16", "bf16", "f32"])
    if kind == "vq":
        return {"kind": kind, "rows": 8 * _log(rng, 64, 1280), "cols": 128 * _log(rng, 8, 80),
                "mats": rng.randint(1, 3), "ncols": rng.choice([1, 1, rng.randint(2, 8), rng.randint(2, 16)]), "x": x}
    if kind in ("q6_k", "q8_0"):
        return {"kind": kind, "rows": _log(rng, 500, 20480), "cols": 256 * _log(rng, 4, 40),
                "ncols": rng.choice([1, 1, rng.randint(2, 8)]), "x": x}
    if kind == "prefill":
        return {"kind": kind, "rows": 8 * _log(rng, 64, 1280), "cols": 128 * _log(rng, 8, 80),
                "tokens": _log(rng, 17, 512), "x": x}
    if kind == "decode":
        pos = _log(rng, 20, 30000)
        return {"kind": kind, "tokens": 1, "pos": pos, "max_ctx": rng.choice([c for c in (1024, 8192, 32768) if c > pos]),
                "x": x}
    if kind == "verify":
        pos = _log(rng, 20, 16000)
        return {"kind": kind, "tokens": rng.randint(2, 8), "pos": pos,
                "max_ctx": rng.choice([c for c in (1024, 8192, 32768) if c > pos + 8]), "x": x}
    pos = rng.choice([0, _log(rng, 16, 16000)])
    return {"kind": "prompt", "tokens": _log(rng, 3, 512), "pos": pos,
            "max_ctx": rng.choice([c for c in (1024, 8192, 32768) if c > pos + 512]), "x": x}


# ---------------------------------------------------------------- inputs


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) + salt)


def _x(case, seed, salt, n, cols):
    """Activations a matvec reads: a norm's output, or an FFN's gelu(gate) * up."""
    g = _gen(seed, salt)
    x = torch.randn(n, cols, generator=g, device="cuda")
    if cols == FFN:
        x = torch.nn.functional.gelu(x) * torch.randn(n, cols, generator=g, device="cuda")
    return x if case["x"] == "f32" else x.to(torch.bfloat16)


def _containers(seed, shapes):
    def one(i):
        return sm.synth_container(10007 * (seed + 1) + i, *shapes[i])
    with concurrent.futures.ThreadPoolExecutor(8) as ex:
        return list(ex.map(one, range(len(shapes))))


def _q8_0(seed, salt, rows, cols):
    """Q8_0 blocks on the GPU: uniform quants, positive scales of a trained head's size."""
    g = _gen(seed, salt)
    n = rows * (cols // 32)
    b = torch.randint(0, 256, (n, 34), generator=g, device="cuda", dtype=torch.uint8)
    b[:, :2] = (1e-4 + 9e-4 * torch.rand(n, 1, generator=g, device="cuda")).to(torch.float16).view(torch.uint8)
    return b.view(-1)


def _q6_k(seed, salt, rows, cols):
    return torch.from_numpy(sm.synth_q6k(10007 * (seed + 1) + salt, rows, cols)).cuda()


def _q6k_shapes():
    """One layer of the Q6_K trunk; matrices that share x are stacked by rows."""
    return (("qkvg", QD + 2 * KVD + HEADS, HIDDEN), ("out", HIDDEN, QD), ("gate_up", 2 * FFN, HIDDEN),
            ("down", HIDDEN, FFN))


class _Rows:
    """The rows of a model's cache, for torch.as_tensor: tensors over them
    hold this object, and with it the model whose memory they show."""

    def __init__(self, model, ptr, shape):
        self.model = model
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def _model_inputs(case, seed):
    hosts = _containers(seed, [(r, c) for _ in range(LAYERS) for _, r, c in LAYER_MATS])
    g = _gen(seed, 1)
    norms = 1 + 0.1 * torch.randn(2 * LAYERS + 1, HIDDEN, generator=g, device="cuda")
    head = _q8_0(seed, 2, VOCAB, HIDDEN)
    # cached keys and values of the size that this model's own projections give
    cache = [[1.5 * torch.randn(case["pos"], KVD, generator=g, device="cuda") for _ in range(2)] for _ in range(LAYERS)]
    tokens = np.random.default_rng(seed).integers(0, VOCAB, case["tokens"]).tolist()
    return hosts, norms, head, cache, tokens


def prepare(case, seed):
    kind = case["kind"]
    if kind == "vq":
        mats = [sm.DeviceContainer(h) for h in _containers(seed, [(case["rows"], case["cols"])] * case["mats"])]
        x = _x(case, seed, 3, case["ncols"], case["cols"])
        ys = [torch.zeros(case["ncols"], case["rows"], device="cuda") for _ in mats]
        return {"case": case, "mats": mats, "x": x, "ys": ys}
    if kind in ("q6_k", "q8_0"):
        blocks = (_q6_k if kind == "q6_k" else _q8_0)(seed, 4, case["rows"], case["cols"])
        return {"case": case, "blocks": blocks, "x": _x(case, seed, 3, case["ncols"], case["cols"]),
                "y": torch.zeros(case["ncols"], case["rows"], device="cuda")}
    if kind == "q6k-layer":
        plan, ys, keep = sm.Plan(), [], []
        for i, (_, rows, cols) in enumerate(_q6k_shapes()):
            b, x = _q6_k(seed, 10 + i, rows, cols), _x(case, seed, 20 + i, case["ncols"], cols)
            y = torch.zeros(case["ncols"], rows, device="cuda")
            plan.add_kquant("q6_k", b, rows, cols, x, y, ncols=case["ncols"])
            keep.append((b, x))
            ys.append(y)
        plan.run()
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        plan.capture(stream)
        torch.cuda.synchronize()
        return {"case": case, "plan": plan, "ys": ys, "keep": keep}
    if kind == "prefill":
        m = sm.DeviceContainer(_containers(seed, [(case["rows"], case["cols"])])[0])
        return {"case": case, "mat": m, "x": _x(case, seed, 3, case["tokens"], case["cols"]),
                "y": torch.zeros(case["tokens"], case["rows"], device="cuda")}
    hosts, norms, head, cache, tokens = _model_inputs(case, seed)
    cfg = dict(hidden=HIDDEN, layers=LAYERS, heads=HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM, intermediate=FFN,
               vocab=VOCAB, eps=EPS, sliding_window=WINDOW, rope_full_theta=ROPE[1][0], rope_full_partial=ROPE[1][1],
               rope_slide_theta=ROPE[0][0], rope_slide_partial=ROPE[0][1], max_ctx=case["max_ctx"],
               x_dtype=sm.X_F32 if case["x"] == "f32" else sm.X_BF16, dim=4, nc=4096, nstages=2, v3=1)
    layers = []
    for li in range(LAYERS):
        L = {name: sm.DeviceContainer(hosts[6 * li + i]) for i, (name, _, _) in enumerate(LAYER_MATS)}
        layers.append(dict(L, in_norm=norms[2 * li], post_norm=norms[2 * li + 1], full=li % 4 == 3))
    model = sm.Model(cfg, layers, head, norms[2 * LAYERS])
    pos, n, rows = case["pos"], case["tokens"], []
    for li in range(LAYERS):
        for ptr, old in zip(model.kv(li), cache[li]):
            t = torch.as_tensor(_Rows(model, ptr, (case["max_ctx"], KVD)), device="cuda")
            t[:pos] = old
            rows.append(t[pos:pos + n])
    logits = torch.zeros((n, VOCAB) if kind == "verify" else VOCAB, device="cuda")
    state = {"case": case, "model": model, "tokens": tokens, "logits": logits, "rows": rows}
    if kind == "decode":
        model.forward(tokens[0], pos, logits)
        state["stream"] = torch.cuda.Stream()
        state["stream"].wait_stream(torch.cuda.current_stream())
        model.capture(logits, state["stream"])
    else:
        model.reserve(max(8, n))
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "vq":
        mats, x, ys = state["mats"], state["x"], state["ys"]
        if len(mats) == 1:
            mats[0].gemv(x, ys[0], ncols=case["ncols"])
        else:
            sm.gemv_multi(mats, x, ys, ncols=case["ncols"])
        return ys
    if kind in ("q6_k", "q8_0"):
        sm.kquant_gemv(kind, state["blocks"], case["rows"], case["cols"], state["x"], state["y"], ncols=case["ncols"])
        return state["y"]
    if kind == "q6k-layer":
        state["plan"].launch()
        return state["ys"]
    if kind == "prefill":
        state["mat"].prefill(state["x"], state["y"])
        return state["y"]
    m, tokens, pos, logits = state["model"], state["tokens"], case["pos"], state["logits"]
    if kind == "decode":
        m.replay(tokens[0], pos, torch.cuda.current_stream())
    elif kind == "verify":
        m.verify(tokens, pos, logits)
    else:
        m.forward_batch(tokens, pos, logits)
    return {"logits": logits, "kv": state["rows"]}


# ---------------------------------------------------------------- costs


def _vq_bytes(rows, cols):
    return sm.lib().sparkmv_stage_bytes(1, rows, cols, 4, 4096) * 2


def work(case):
    kind, xb = case["kind"], 4 if case["x"] == "f32" else 2
    if kind in ("vq", "q6_k", "q8_0", "prefill"):
        rows, cols = case["rows"] * case.get("mats", 1), case["cols"]
        n = case["tokens"] if kind == "prefill" else case["ncols"]
        if kind == "q6_k":
            w = rows * (cols // 256) * 210
        elif kind == "q8_0":
            w = rows * (cols // 32) * 34
        else:
            w = _vq_bytes(case["rows"], cols) * case.get("mats", 1)
        return {"bytes": w + n * cols * xb + n * rows * 4, "flops": 2 * n * rows * cols}
    if kind == "q6k-layer":
        n = case["ncols"]
        return {"bytes": sum(r * (c // 256) * 210 + n * c * xb + n * r * 4 for _, r, c in _q6k_shapes()),
                "flops": sum(2 * n * r * c for _, r, c in _q6k_shapes())}
    n, pos = case["tokens"], case["pos"]
    heads = n if kind == "verify" else 1        # rows of logits
    nbytes = sum(_vq_bytes(r, c) for _, r, c in LAYER_MATS) * LAYERS + VOCAB * (HIDDEN // 32) * 34 + heads * VOCAB * 4
    flops = 2 * n * sum(r * c for _, r, c in LAYER_MATS) * LAYERS + 2 * heads * VOCAB * HIDDEN
    for li in range(LAYERS):
        window = 10**9 if li % 4 == 3 else WINDOW
        span = pos + n - max(0, pos + 1 - window)     # cached positions read, and the new rows written
        seen = sum(min(p + 1, window) for p in range(pos, pos + n))
        nbytes += 2 * KVD * 4 * (span + n)
        flops += 4 * HEAD_DIM * HEADS * seen
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from `exact` that the paths show."""
    kind = case["kind"]
    if kind in ("vq", "q6_k", "q8_0", "q6k-layer"):
        # products of f16 weights and f16 (or hi + lo f16) activations, f32 sums
        return {"rel": 2e-6}
    if kind == "prefill":
        # the folded weight, and f32 activations, are rounded to f16
        return {"rel": 1.5e-3}
    if case["x"] == "bf16":
        # activations rounded to bf16 before each of the 20 matvecs of the four layers
        return {"rel": 4e-2}
    # f32 activations: what shows is the last bit of the rope angles, which a
    # late position multiplies; longer chunks round activations to f16
    return {"rel": 5e-3 if kind != "prompt" or case["tokens"] <= 16 else 1e-2}


# ------------------------------------------------------- the same in 64 bits


def _vq_weight(host, rows, cols):
    """An RQVQ container's matrix in f64, from its bytes: per stage a 24-byte
    header, 4096 x 4 f16 codewords, f16 row gains, 12-bit indices."""
    data = torch.from_numpy(np.ascontiguousarray(host)).cuda()
    per = 24 + 4096 * 8 + 2 * rows + rows * (cols // 4 * 12 // 8)
    start = data.numel() - 2 * per
    W = torch.zeros(rows, cols, dtype=torch.float64, device="cuda")
    for s in range(2):
        p = data[start + s * per:start + (s + 1) * per].clone()
        cb = p[24:24 + 32768].clone().view(torch.float16).view(4096, 4).double()
        gains = p[24 + 32768:24 + 32768 + 2 * rows].clone().view(torch.float16).double()
        b = p[24 + 32768 + 2 * rows:].view(rows, cols // 8, 3).to(torch.int64)
        idx = torch.stack([b[..., 0] | (b[..., 1] & 15) << 8, b[..., 1] >> 4 | b[..., 2] << 4], dim=-1).view(rows, -1)
        W += cb[idx].view(rows, cols) * gains[:, None]
    return W


def _q8_0_weight(blocks, rows, cols):
    b = blocks.view(rows, cols // 32, 34)
    d = b[..., :2].contiguous().view(torch.float16).double()
    return (d * b[..., 2:].contiguous().view(torch.int8).double()).view(rows, cols)


def _q6_k_weight(blocks, rows, cols):
    b = blocks.view(rows, cols // 256, 210)
    ql, qh = b[..., :128].to(torch.int64), b[..., 128:192].to(torch.int64)
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    d = b[..., 208:].contiguous().view(torch.float16).double()
    parts = []
    for half in range(2):
        lo, hi, h = ql[..., 64 * half:64 * half + 32], ql[..., 64 * half + 32:64 * half + 64], qh[..., 32 * half:32 * half + 32]
        parts += [(lo & 15) | (h & 3) << 4, (hi & 15) | (h >> 2 & 3) << 4, lo >> 4 | (h >> 4 & 3) << 4,
                  hi >> 4 | (h >> 6 & 3) << 4]
    q = torch.cat(parts, dim=-1).double() - 32
    return (q * sc.repeat_interleave(16, dim=-1) * d).view(rows, cols)


def _norm(h, w):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos0, full):
    """The first rotated elements of every head turned by their position; the
    angles are f32 by definition (a late position's differ visibly in 64 bits)."""
    theta, share = ROPE[int(full)]
    dim = int(HEAD_DIM * share)
    half = dim // 2
    inv = 1 / (theta ** (torch.arange(half, dtype=torch.float64, device="cuda") * 2 / dim)).float()
    a = ((pos0 + torch.arange(x.shape[0], device="cuda").float())[:, None] * inv).double()
    c, s = a.cos()[:, None], a.sin()[:, None]
    x0, x1 = x[..., :half], x[..., half:dim]
    return torch.cat([x0 * c - x1 * s, x1 * c + x0 * s, x[..., dim:]], dim=-1)


def _exact_model(case, seed):
    hosts, norms, head, cache, tokens = _model_inputs(case, seed)
    n, pos = case["tokens"], case["pos"]
    hw = _q8_0_weight(head, VOCAB, HIDDEN)
    h = hw[torch.tensor(tokens, device="cuda")]
    at = torch.arange(pos, pos + n, device="cuda")[:, None]
    rows = []
    for li in range(LAYERS):
        W = {name: _vq_weight(hosts[6 * li + i], r, c) for i, (name, r, c) in enumerate(LAYER_MATS)}
        full = li % 4 == 3
        x = _norm(h, norms[2 * li])
        qkv, gate = x @ W["qkv"].T, torch.sigmoid(x @ W["attn_gate"].T)
        q = _rope(qkv[:, :QD].view(n, HEADS, HEAD_DIM), pos, full)
        k = _rope(qkv[:, QD:QD + KVD].view(n, KV_HEADS, HEAD_DIM), pos, full)
        v = qkv[:, QD + KVD:]
        rows += [k.reshape(n, KVD), v]
        first = 0 if full else max(0, pos + 1 - WINDOW)
        K = torch.cat([cache[li][0][first:].double(), k.reshape(n, KVD)]).view(-1, KV_HEADS, HEAD_DIM)
        V = torch.cat([cache[li][1][first:].double(), v]).view(-1, KV_HEADS, HEAD_DIM)
        seen = torch.arange(first, pos + n, device="cuda")[None]
        hidden = (seen > at) | (False if full else seen <= at - WINDOW)
        out = torch.empty(n, HEADS, HEAD_DIM, dtype=torch.float64, device="cuda")
        for i in range(HEADS):
            kv = i // (HEADS // KV_HEADS)
            s = (q[:, i] @ K[:, kv].T.contiguous() / math.sqrt(HEAD_DIM)).masked_fill(hidden, -math.inf)
            out[:, i] = torch.softmax(s, dim=-1) @ V[:, kv].contiguous() * gate[:, i:i + 1]
        h = h + out.view(n, QD) @ W["out"].T
        x = _norm(h, norms[2 * li + 1])
        h = h + (torch.nn.functional.gelu(x @ W["gate"].T) * (x @ W["up"].T)) @ W["down"].T
    h = _norm(h if case["kind"] == "verify" else h[-1], norms[2 * LAYERS])
    return {"logits": h @ hw.T, "kv": rows}


def exact(case, seed):
    kind = case["kind"]
    if kind == "vq":
        x = _x(case, seed, 3, case["ncols"], case["cols"]).double()
        hosts = _containers(seed, [(case["rows"], case["cols"])] * case["mats"])
        return [x @ _vq_weight(h, case["rows"], case["cols"]).T for h in hosts]
    if kind in ("q6_k", "q8_0"):
        x = _x(case, seed, 3, case["ncols"], case["cols"]).double()
        make, weight = (_q6_k, _q6_k_weight) if kind == "q6_k" else (_q8_0, _q8_0_weight)
        return x @ weight(make(seed, 4, case["rows"], case["cols"]), case["rows"], case["cols"]).T
    if kind == "q6k-layer":
        return [_x(case, seed, 20 + i, case["ncols"], c).double() @ _q6_k_weight(_q6_k(seed, 10 + i, r, c), r, c).T
                for i, (_, r, c) in enumerate(_q6k_shapes())]
    if kind == "prefill":
        host = _containers(seed, [(case["rows"], case["cols"])])[0]
        return _x(case, seed, 3, case["tokens"], case["cols"]).double() @ _vq_weight(host, case["rows"], case["cols"]).T
    return _exact_model(case, seed)
