"""The calls a program makes of this framework, at the sizes it makes them.

A program that runs a model over strataflow_amd owns a paged KV cache, per
layer weights and a page table, and calls per layer: the Q/K/V product with
RoPE and the append (``qkv``), the attention of a decode step (``decode``,
``window``) or of a prompt chunk (``prefill``), a dense product with the
residual (``product``), and the ffn norm, routing and experts (``moe``).
``tiny`` is the whole forward of the repository's own tiny MoE model.

Shapes: ``mixtral`` is the shape of the repository's benchmark (32 query
heads, 8 kv heads, head_dim 128, n_embd 4096, n_ff 14336, 8 experts, 2 used),
``half`` a generic model of half its width, ``tiny`` the tiny MoE model's.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from strataflow_amd import layer as ops
from strataflow_amd import synth
from strataflow_amd.paged_kv import SFA_KV_F16, SFA_KV_F32, SFA_KV_Q8_0, PagedKV
from strataflow_amd.pager import SFA_ATTEND_WINDOW, KvPager
from strataflow_amd.tiny_moe import TinyMoeConfig, TinyMoeGpu, TinyMoeWeights

DEV = "cuda"
PAGE = 256
FREQ = 1e6
EPS = 1e-5
KV = {"f32": SFA_KV_F32, "f16": SFA_KV_F16, "q8_0": SFA_KV_Q8_0}
ROW = {"f32": 4.0, "f16": 2.0, "q8_0": 34.0 / 32.0}  # cache bytes an element
WT = {"f32": torch.float32, "f16": torch.float16}
# query heads, kv heads, head_dim, n_embd, n_ff, experts, used
SHAPES = {
    "mixtral": (32, 8, 128, 4096, 14336, 8, 2),
    "half": (16, 4, 128, 2048, 5632, 16, 2),
    "tiny": (8, 4, 32, 256, 512, 8, 2),
}
# the dense products of those layers: (n_in, n_out)
PRODUCTS = {"mixtral": (4096, 4096), "half": (2048, 2048), "tiny": (256, 256), "head": (4096, 32000)}


def listed():
    return [
        # one greedy token of the tiny model: the smallest whole call, launches and latency
        {"name": "tiny_token", "op": "tiny", "pos0": 95, "n_tok": 1},
        # one decode step of one conversation at the benchmark's context
        {"name": "decode_f16_b1", "op": "decode", "kv": "f16", "shape": "mixtral", "lens": "4096"},
        # a serving batch of long conversations over a quantised cache
        {"name": "decode_q8_0_b8", "op": "decode", "kv": "q8_0", "shape": "mixtral",
         "lens": "8211,30720,12001,25333,17000,32768,9999,21470"},
        # a step of four long chats under the sliding window, the append in it
        {"name": "window_f16_b4", "op": "window", "kv": "f16", "shape": "mixtral", "window": 4096,
         "lens": "9000,5121,12288,7777"},
        # the second half of a 4096-token prompt
        {"name": "prefill_f16_2048", "op": "prefill", "kv": "f16", "shape": "mixtral", "past": 2048, "n_tok": 2048},
        # a chat turn: a short question on a long history
        {"name": "prefill_f16_turn", "op": "prefill", "kv": "f16", "shape": "mixtral", "past": 8100, "n_tok": 93},
        # a ragged prompt chunk over a quantised cache
        {"name": "prefill_q8_0_chunk", "op": "prefill", "kv": "q8_0", "shape": "mixtral", "past": 3000, "n_tok": 777},
        # a prompt chunk's Q/K/V product, RoPE and append
        {"name": "qkv_chunk", "op": "qkv", "kv": "f16", "shape": "mixtral", "wt": "f16", "past": 1000, "n_tok": 512},
        # the attention's output product with the residual, for a batch of decoding sequences
        {"name": "product_b16", "op": "product", "dims": "mixtral", "wt": "f16", "n_tok": 16},
        # the ffn half of a layer: one decoding sequence, a batch of them, a prompt chunk
        {"name": "moe_token", "op": "moe", "shape": "mixtral", "n_tok": 1},
        {"name": "moe_b13", "op": "moe", "shape": "mixtral", "n_tok": 13},
        {"name": "moe_chunk", "op": "moe", "shape": "mixtral", "n_tok": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["tiny", "decode", "decode", "window", "prefill", "prefill", "qkv", "product", "moe", "moe"])
    if op == "tiny":
        n = rng.choice([1, _log(rng, 2, 128)])
        return {"op": op, "pos0": rng.randint(1, 300), "n_tok": n}
    if op == "decode":
        kv = rng.choice(["f16", "f16", "q8_0", "f32"])
        batch = _log(rng, 1, 32)
        top = min(32768, {"f16": 90000, "q8_0": 158000, "f32": 45000}[kv] // batch)
        lens = [_log(rng, 32, top) for _ in range(batch)]
        return {"op": op, "kv": kv, "shape": rng.choice(["mixtral", "half"]), "lens": ",".join(map(str, lens))}
    if op == "window":
        lens = [_log(rng, 300, 14000) for _ in range(_log(rng, 1, 8))]
        return {"op": op, "kv": rng.choice(["f16", "f32"]), "shape": rng.choice(["mixtral", "half"]),
                "window": 256 * rng.randint(2, 16), "lens": ",".join(map(str, lens))}
    if op == "prefill":
        kv = rng.choice(["f16", "f16", "q8_0", "f32"])
        n = _log(rng, 8, 2048)
        past = rng.randint(0, 2048) if n > 700 else rng.randint(0, 8192)
        return {"op": op, "kv": kv, "shape": rng.choice(["mixtral", "half"]), "past": past, "n_tok": n}
    if op == "qkv":
        return {"op": op, "kv": rng.choice(["f16", "f32"]), "shape": rng.choice(["mixtral", "half", "tiny"]),
                "wt": rng.choice(["f16", "f16", "f32"]), "past": rng.randint(0, 4000), "n_tok": _log(rng, 1, 512)}
    if op == "product":
        return {"op": op, "dims": rng.choice(sorted(PRODUCTS)), "wt": rng.choice(["f16", "f16", "f32"]),
                "n_tok": _log(rng, 1, 512)}
    return {"op": op, "shape": rng.choice(["mixtral", "half"]), "n_tok": _log(rng, 1, 512)}


# ---- inputs, from the seed alone ------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    t = torch.randn(shape, generator=g, device=DEV, dtype=dtype)
    return t if std == 1.0 else t.mul_(std)


def _lens(case):
    return [int(n) for n in case["lens"].split(",")]


def _attn_inputs(case, seed):
    """Histories, queries and (window) the step's new K/V rows."""
    hq, hkv, hd = SHAPES[case["shape"]][:3]
    g = _gen(seed)
    if case["op"] == "prefill":
        lens, n_q = [case["past"] + case["n_tok"]], case["n_tok"]
    else:
        lens, n_q = _lens(case), len(_lens(case))
    hist = [(_randn(g, n, hkv, hd), _randn(g, n, hkv, hd)) for n in lens]
    return lens, hist, _randn(g, n_q, hq, hd)


def _qkv_inputs(case, seed):
    hq, hkv, hd, n_embd = SHAPES[case["shape"]][:4]
    g = _gen(seed)
    w = _randn(g, (hq + 2 * hkv) * hd, n_embd, dtype=WT[case["wt"]], std=n_embd ** -0.5)
    return w, _randn(g, case["n_tok"], n_embd)  # x: a normed row


def _product_inputs(case, seed):
    n_in, n_out = PRODUCTS[case["dims"]]
    g = _gen(seed)
    w = _randn(g, n_out, n_in, dtype=WT[case["wt"]], std=n_in ** -0.5)
    return w, _randn(g, case["n_tok"], n_in), _randn(g, case["n_tok"], n_out)


def _moe_inputs(case, seed):
    _, _, _, n_embd, n_ff, n_exp, _ = SHAPES[case["shape"]]
    g = _gen(seed)
    h = torch.float16
    return {
        "x": _randn(g, case["n_tok"], n_embd, std=2.0),
        "norm": 1.0 + 0.1 * _randn(g, n_embd),
        "router": _randn(g, n_exp, n_embd, dtype=h, std=n_embd ** -0.5),
        "gate": _randn(g, n_exp, n_ff, n_embd, dtype=h, std=n_embd ** -0.5),
        "up": _randn(g, n_exp, n_ff, n_embd, dtype=h, std=n_embd ** -0.5),
        "down": _randn(g, n_exp, n_embd, n_ff, dtype=h, std=n_ff ** -0.5),
    }


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(DEV)


def _cache(case, lens, seed):
    hq, hkv, hd = SHAPES[case["shape"]][:3]
    n_pages = sum(-(-n // PAGE) for n in lens) + 2
    kv = PagedKV(1, hq, hkv, hd, KV[case["kv"]], PAGE, n_pages)
    return kv, _i32(synth.page_tables(np.random.default_rng(seed), lens, PAGE, n_pages))


def prepare(case, seed):
    """What the program has before the call: the cache with its history, page
    tables, weights, inputs and the output buffers a decode loop keeps."""
    op = case["op"]
    if op == "tiny":
        cfg = TinyMoeConfig()
        m = TinyMoeGpu(cfg, TinyMoeWeights(cfg, seed), 512, seed=seed)
        toks = np.random.default_rng(seed).integers(0, cfg.n_vocab, case["pos0"] + case["n_tok"])
        m.forward(toks[:case["pos0"]], 0)
        return {"op": op, "model": m, "tokens": toks[case["pos0"]:], "pos0": case["pos0"]}
    if op in ("decode", "prefill"):
        lens, hist, q = _attn_inputs(case, seed)
        kv, pt = _cache(case, lens, seed)
        for b, (k, v) in enumerate(hist):
            n = lens[b]
            kv.append(0, k, v, torch.full((n,), b, dtype=torch.int32, device=DEV),
                      torch.arange(n, dtype=torch.int32, device=DEV), pt)
        st = {"op": op, "kv": kv, "q": q, "pt": pt, "past": case.get("past", 0),
              "seq_len": _i32(lens), "max_len": max(lens),
              "out": torch.empty((q.shape[0], q.shape[1] * q.shape[2]), device=DEV)}
        if op == "decode":
            kv.workspace(len(lens), st["max_len"])
        else:
            st["pt"] = pt[0]
        return st
    if op == "window":
        hq, hkv, hd = SHAPES[case["shape"]][:3]
        lens, hist, q = _attn_inputs(case, seed)
        pager = KvPager(n_layer=1, n_head=hq, n_head_kv=hkv, head_dim=hd, kv_type=KV[case["kv"]], page_size=PAGE,
                        n_seq=len(lens), n_ctx=max(lens) + 1, window=case["window"], attend=SFA_ATTEND_WINDOW,
                        seed=seed)
        used = [0] * len(lens)
        while True:  # the prompt, a page of each sequence at a time; the last position is the step's
            n_tok = [min(PAGE, n - 1 - u) for n, u in zip(lens, used)]
            if not any(n_tok):
                break
            assert pager.begin(n_tok) == 0
            parts = [(k[u:u + t], v[u:u + t]) for (k, v), u, t in zip(hist, used, n_tok)]
            pager.append(0, torch.cat([k for k, _ in parts]), torch.cat([v for _, v in parts]))
            used = [u + t for u, t in zip(used, n_tok)]
        assert pager.begin([1] * len(lens)) == 0
        return {"op": op, "pager": pager, "q": q, "k": torch.cat([k[-1:] for k, _ in hist]),
                "v": torch.cat([v[-1:] for _, v in hist]),
                "out": torch.empty((q.shape[0], q.shape[1] * q.shape[2]), device=DEV)}
    if op == "qkv":
        w, x = _qkv_inputs(case, seed)
        n, end = case["n_tok"], case["past"] + case["n_tok"]
        kv, pt = _cache(case, [end], seed)
        return {"op": op, "kv": kv, "w": w, "x": x, "pt": pt,
                "seq": torch.zeros(n, dtype=torch.int32, device=DEV),
                "pos": torch.arange(case["past"], end, dtype=torch.int32, device=DEV),
                "q": torch.empty((n, kv.n_head, kv.head_dim), device=DEV),
                "ctype": {"f16": torch.float16, "f32": torch.float32}[case["kv"]]}
    if op == "product":
        w, x, res = _product_inputs(case, seed)
        return {"op": op, "w": w, "x": x, "res": res, "out": torch.empty_like(res)}
    st = _moe_inputs(case, seed)
    n_embd, n_ff, used = SHAPES[case["shape"]][3], SHAPES[case["shape"]][4], SHAPES[case["shape"]][6]
    n = case["n_tok"]
    st.update(op=op, used=used, cur=torch.empty((n, n_embd), device=DEV), out=torch.empty((n, n_embd), device=DEV),
              ids=torch.empty((n, used), dtype=torch.int32, device=DEV), wts=torch.empty((n, used), device=DEV),
              ws=torch.empty(n * used * n_ff * 4, dtype=torch.uint8, device=DEV))
    return st


def run(st):
    op = st["op"]
    if op == "tiny":
        return st["model"].forward(st["tokens"], st["pos0"])
    if op == "decode":
        return st["kv"].decode(0, st["q"], st["pt"], st["seq_len"], st["max_len"], out=st["out"])
    if op == "prefill":
        return st["kv"].prefill(0, st["q"], st["pt"], st["past"], out=st["out"])
    if op == "window":
        return st["pager"].append_attend(0, st["k"], st["v"], st["q"], out=st["out"])
    if op == "qkv":
        q = st["kv"].qkv_rope_append(0, st["w"], st["x"], st["seq"], st["pos"], st["pt"], FREQ, q=st["q"])
        return q, st["kv"].k[0].view(st["ctype"]), st["kv"].v[0].view(st["ctype"])
    if op == "product":
        return ops.mul_mat_vec(st["w"], st["x"], residual=st["res"], out=st["out"])
    cur, ids, wts = ops.moe_norm_gate(st["x"], st["norm"], EPS, st["router"], st["used"], out=st["cur"],
                                      ids=st["ids"], weights=st["wts"])
    y = ops.moe_ffn(cur, st["x"], ids, wts, st["gate"], st["up"], st["down"], out=st["out"], workspace=st["ws"])
    return cur, ids, wts, y


# ---- the work a pass cannot do without ------------------------------------------

def _experts_read(n_exp, used, n_tok):
    return n_exp * (1.0 - (1.0 - used / n_exp) ** n_tok)  # expected, routing near uniform


def work(case):
    op, n = case["op"], case.get("n_tok", 1)
    if op == "tiny":
        c = TinyMoeConfig()
        attn = (2 * c.n_head + 2 * c.n_head_kv) * c.head_dim * c.n_embd
        exp = 3 * c.n_embd * c.n_ff
        layer_w = attn + c.n_expert * c.n_embd + exp * _experts_read(c.n_expert, c.n_expert_used, n)
        ctx = case["pos0"] + n
        kv = 2 * ctx * c.n_head_kv * c.head_dim * 2
        pairs = n * case["pos0"] + n * (n + 1) / 2
        flops = 2 * n * (attn + c.n_expert * c.n_embd + exp * c.n_expert_used) + 4 * c.head_dim * c.n_head * pairs
        return {"bytes": c.n_layer * (4 * layer_w + kv) + 4 * c.n_vocab * (c.n_embd + 1) + 4 * n * c.n_embd,
                "flops": c.n_layer * flops + 2 * c.n_vocab * c.n_embd}
    if op == "product":
        n_in, n_out = PRODUCTS[case["dims"]]
        return {"bytes": n_in * n_out * WT[case["wt"]].itemsize + 4 * n * (n_in + 2 * n_out),
                "flops": 2 * n * n_in * n_out}
    hq, hkv, hd, n_embd, n_ff, n_exp, used = SHAPES[case["shape"]]
    if op == "qkv":
        rows = (hq + 2 * hkv) * hd
        return {"bytes": rows * n_embd * WT[case["wt"]].itemsize
                + n * (4 * n_embd + 4 * hq * hd + 2 * hkv * hd * ROW[case["kv"]]),
                "flops": 2 * n * rows * n_embd}
    if op == "moe":
        read = _experts_read(n_exp, used, n)
        return {"bytes": 2 * (3 * n_embd * n_ff * read + n_exp * n_embd) + n * (4 * 3 * n_embd + 8 * used),
                "flops": 2 * n * (3 * n_embd * n_ff * used + n_exp * n_embd)}
    row = 2 * hkv * hd * ROW[case["kv"]]  # K and V of one position
    if op == "prefill":
        pairs = n * case["past"] + n * (n + 1) / 2
        return {"bytes": (case["past"] + n) * row + 2 * 4 * n * hq * hd, "flops": 4 * hd * hq * pairs}
    lens = _lens(case)
    span = sum(lens) if op == "decode" else sum(min(m, case["window"]) for m in lens)
    new = len(lens) * 2 * 4 * hkv * hd if op == "window" else 0
    return {"bytes": span * row + new + 2 * 4 * len(lens) * hq * hd, "flops": 4 * hd * hq * span}


def tolerance(case):
    op = case["op"]
    if op == "tiny":  # f32 weights, an f16 cache: a cache rounding moved by a last ulp travels through four layers
        return {"rel": 5e-4, "max": 5e-3}
    if op in ("decode", "window", "prefill"):
        # f32: sums in another order. f16: probabilities rounded to f16 at other references of the running
        # maximum, as the split of the positions moves them. q8_0 takes the same probabilities.
        return {"rel": 2e-5, "max": 2e-4} if case["kv"] == "f32" else {"rel": 1.5e-3, "max": 1.5e-2}
    if op == "qkv":
        # q: sums in another order; cached f16 rows: a last-ulp difference moves a few roundings
        return {"rel": 1e-4, "max": 2e-3}
    if op == "product":
        return {"rel": 1e-5, "max": 1e-4}
    # the activation is rounded to f16 before the down product: a last-ulp difference moves a few of them
    return {"rel": 1e-4, "max": 1e-3, "differ": 0.0}


# ---- the same in 64 bits --------------------------------------------------------
# Operands as the entry points document them: F16 weights take the activation
# rounded to f16, a cache holds what its type holds.

def _cached(x, kv):
    if kv == "f32":
        return x.double()
    if kv == "f16":
        return x.half().double()
    b = x.reshape(*x.shape[:-1], x.shape[-1] // 32, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    q = torch.where(d > 0, b / torch.where(d > 0, d, torch.ones_like(d)), torch.zeros_like(b))
    q = torch.sign(q) * torch.floor(q.abs() + 0.5)
    return (q.double() * d.half().double()).reshape(x.shape)


def _attend(q, k, v, first):
    """q [T, Hq, hd]; k, v [n, Hkv, hd] in 64 bits; row t attends 0..first + t."""
    T, hq, hd = q.shape
    n, hkv = k.shape[:2]
    out = torch.empty((T, hq, hd), dtype=torch.float64, device=q.device)
    mask = torch.arange(n, device=q.device)[None, :] > first + torch.arange(T, device=q.device)[:, None]
    for h in range(hq):
        kh, vh = k[:, h // (hq // hkv)].contiguous(), v[:, h // (hq // hkv)].contiguous()
        s = (q[:, h].double() @ kh.t()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), -1) @ vh
    return out.reshape(T, hq * hd)


def _rope(x, pos, base):
    """RoPE of adjacent pairs at ggml's f32 thetas (theta *= base^(-2/hd))."""
    hd = x.shape[-1]
    scale = float(synth.powf(np.float32(base), np.float32(-2.0) / np.float32(hd)))
    th = [pos.float()]
    for _ in range(hd // 2 - 1):
        th.append(th[-1] * scale)
    th = torch.stack(th, -1).double()[:, None, :]
    c, s = torch.cos(th), torch.sin(th)
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * c - x1 * s, x0 * s + x1 * c), -1).reshape(x.shape)


def _operand(x, w):
    return x.half().double() if w.dtype == torch.float16 else x.double()


def _rms(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _route(logits, used):
    p = torch.softmax(logits, -1)
    w, ids = torch.sort(p, dim=-1, descending=True, stable=True)
    w, ids = w[:, :used], ids[:, :used]
    return ids, w / w.sum(-1, keepdim=True).clamp_min(6.103515625e-5)


def _experts(x, res, ids, wts, gate, up, down):
    y = torch.zeros_like(res)
    for e in range(gate.shape[0]):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        if t.numel() == 0:
            continue
        xe = _operand(x[t], gate)
        g, u = xe @ gate[e].double().t(), xe @ up[e].double().t()
        act = _operand(g / (1.0 + torch.exp(-g)) * u, down)
        y.index_add_(0, t, (act @ down[e].double().t()) * wts[t, j][:, None])
    return y + res


def _exact_tiny(case, seed):
    c = TinyMoeConfig()
    w = TinyMoeWeights(c, seed)
    n = case["pos0"] + case["n_tok"]
    toks = np.random.default_rng(seed).integers(0, c.n_vocab, n)

    def d(a):
        return torch.from_numpy(a).to(DEV).double()

    pos = torch.arange(n, device=DEV)
    x = d(w.token_embd)[torch.from_numpy(toks).to(DEV)]
    for L in w.layers:
        L = {k: d(a) for k, a in L.items()}
        cur = _rms(x, L["attn_norm"])
        q = _rope((cur @ L["wq"].t()).view(n, c.n_head, c.head_dim), pos, c.freq_base)
        k = _rope((cur @ L["wk"].t()).view(n, c.n_head_kv, c.head_dim), pos, c.freq_base)
        v = (cur @ L["wv"].t()).view(n, c.n_head_kv, c.head_dim)
        x = _attend(q, _cached(k, "f16"), _cached(v, "f16"), 0) @ L["wo"].t() + x
        cur = _rms(x, L["ffn_norm"])
        ids, wts = _route(cur @ L["gate_inp"].t(), c.n_expert_used)
        x = _experts(cur, x, ids, wts, L["gate_exps"], L["up_exps"], L["down_exps"])
    return (_rms(x[-1:], d(w.output_norm)) @ d(w.output).t())[0]


def exact(case, seed):
    op = case["op"]
    if op == "tiny":
        return _exact_tiny(case, seed)
    if op == "qkv":
        hq, hkv, hd = SHAPES[case["shape"]][:3]
        w, x = _qkv_inputs(case, seed)
        n = case["n_tok"]
        y = (_operand(x, w) @ w.double().t()).view(n, hq + 2 * hkv, hd)
        pos = torch.arange(case["past"], case["past"] + n, device=DEV)
        return _rope(y[:, :hq], pos, FREQ), None, None  # the cache's layout is the page table's
    if op == "product":
        w, x, res = _product_inputs(case, seed)
        return _operand(x, w) @ w.double().t() + res.double()
    if op == "moe":
        m = _moe_inputs(case, seed)
        used = SHAPES[case["shape"]][6]
        x = m["x"].double()
        cur = _rms(x, m["norm"].double())
        ids, wts = _route(_operand(cur.float(), m["router"]) @ m["router"].double().t(), used)
        return cur, None, wts, _experts(cur.float(), x, ids, wts, m["gate"], m["up"], m["down"])
    lens, hist, q = _attn_inputs(case, seed)
    if op == "prefill":
        k, v = (_cached(t, case["kv"]) for t in hist[0])
        return _attend(q, k, v, case["past"])
    out = []
    for b, (k, v) in enumerate(hist):
        lo = max(0, lens[b] - case["window"]) if op == "window" else 0
        out.append(_attend(q[b:b + 1], _cached(k[lo:], case["kv"]), _cached(v[lo:], case["kv"]), lens[b] - lo))
    return torch.cat(out)
