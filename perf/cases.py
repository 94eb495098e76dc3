"""The work a serving program has this library do for one attention layer, as
timed cases: decode steps (the newest token of every sequence appended and
attended, `lnskv.device.PagedKV`'s fused calls), prompt chunks (the chunk's K
and V appended, then every chunk token's attention) and the o_proj over Q4_L
weights that follows both (`Q4LMatrix.gemv_accumulate`).

A case names the geometry (query heads, kv heads, head_dim, page type), the
batch (`seqs` sequences whose contexts are drawn from [lo, hi] by the stream
`lens`, so that a case's work does not depend on the seed) and the options of
the call.  The seed makes the values and the order of the pages in the pool.
Stored K and V are N(0, 1) in the page's own type (Q8A: quantised per token
and kv head as the append does), queries N(0, 2^2), so scores have the spread
of a trained layer's rather than a flat softmax.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lns-ml_amd"))
from lnskv import DTYPE_F16, DTYPE_F32, DTYPE_Q8A  # noqa: E402
from lnskv.device import PagedKV, Q4LMatrix, RopeTable  # noqa: E402

PAGE = 16
DTYPES = {"f32": DTYPE_F32, "f16": DTYPE_F16, "q8a": DTYPE_Q8A}
ELEM = {"f32": 4, "f16": 2, "q8a": 1}
THETA = 1.0e7
MAX_BYTES = 2.2e9    # a drawn decode step reads no more than this
MAX_FLOPS = 300e9    # a drawn prompt's attention needs no more than this
DEV = "cuda"


def _attn(name, path, pages, heads, kv_heads, dim, seqs, lo, hi, lens=1, chunk=1, rope=0, gate=False, split=0,
          window=0, copies=0):
    return {"name": name, "path": path, "pages": pages, "heads": heads, "kv_heads": kv_heads, "dim": dim,
            "seqs": seqs, "lo": lo, "hi": hi, "lens": lens, "chunk": chunk, "rope": rope, "gate": gate,
            "split": split, "window": window, "copies": copies}


def listed():
    return [
        # One sequence, one token: the call an interactive engine makes per layer and token, at 4096 tokens of
        # context on the engine's own Q8A pages.  Latency and launches only.
        _attn("call_q8a_4096", "call", "q8a", 32, 8, 128, 1, 4095, 4095),
        # The smallest step: one short sequence, 64-wide heads, f32 pages.
        _attn("step_f32_d64_512", "step", "f32", 32, 4, 64, 1, 512, 512),
        # The Llama-3-8B-shaped layer at batch 32 and ragged contexts, f16 pages: the benchmark's headline step.
        _attn("step_f16_b32", "step", "f16", 32, 8, 128, 32, 512, 4096),
        # A model with 64-wide heads served at an uneven batch of 48, f16 pages.
        _attn("step_f16_d64_b48", "step", "f16", 32, 4, 64, 48, 256, 4096),
        # The batch-32 layer with its cache kept in f32.
        _attn("step_f32_b32", "step", "f32", 32, 8, 128, 32, 512, 4096),
        # The 256-wide gated attention with RoPE (64 of 256) turned in the call, Q8A pages, batch 32.
        _attn("step_q8a_d256_b32", "step", "q8a", 16, 4, 256, 32, 512, 4096, rope=64, gate=True),
        # Long documents: four sequences of 32768 tokens, the caller's own split of 512 tokens.
        _attn("step_f16_32k", "step", "f16", 32, 8, 128, 4, 32768, 32768, split=512),
        # A full server: 136 sequences, some forked, whose tail pages are copied before the step.
        _attn("step_f16_b136", "step", "f16", 32, 8, 128, 136, 256, 8192, copies=8),
        # Chunked prefill of a whole batch: the next 256 prompt tokens of 32 sequences.
        _attn("prompt_f16_b32", "prompt", "f16", 32, 8, 128, 32, 256, 3840, chunk=256, rope=128),
        # One user's prompt: the next 512 tokens of one sequence on Q8A pages, 256-wide heads.
        _attn("prompt_q8a_d256_b1", "prompt", "q8a", 16, 4, 256, 1, 2043, 2043, chunk=512, rope=64),
        # The o_proj after a batch-32 decode step.
        {"name": "o_proj_b32", "path": "o_proj", "rows": 4096, "cols": 4096, "vecs": 32},
        # The o_proj after a 512-token prompt chunk.
        {"name": "o_proj_prompt512", "path": "o_proj", "rows": 4096, "cols": 4096, "vecs": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["step", "step", "step", "prompt", "prompt", "o_proj"])
    if path == "o_proj":
        rows = rng.choice([_log_int(rng, 1000, 8192), 256 * rng.randint(4, 32)])
        return {"path": path, "rows": rows, "cols": 256 * rng.randint(4, 32), "vecs": _log_int(rng, 1, 640)}
    lens = rng.randint(2, 1 << 20)
    if path == "prompt":
        heads, kv, dim = rng.choice([(32, 8, 128), (16, 4, 256), (16, 8, 128), (32, 4, 128), (8, 8, 128)])
        seqs, chunk, hi = _log_int(rng, 1, 32), _log_int(rng, 16, 1024), _log_int(rng, 64, 8192)
        c = _attn("", path, rng.choice(["f16", "q8a"]), heads, kv, dim, seqs, hi // 8, hi, lens, chunk=chunk,
                  rope=rng.choice([0, 64, 128]), window=rng.choice([0, 0, 0, 1024]))
        while work(c)["flops"] > MAX_FLOPS:
            c["hi"], c["chunk"] = max(64, c["hi"] * 3 // 4), max(16, c["chunk"] * 3 // 4)
            c["lo"] = c["hi"] // 8
    else:
        heads, kv, dim = rng.choice([(32, 8, 128), (16, 4, 256), (32, 4, 64), (16, 8, 128), (32, 4, 128), (8, 8, 64)])
        seqs = _log_int(rng, 1, 136)
        hi = _log_int(rng, 256, 32768 if seqs <= 4 else 8192)
        rope, gate = rng.choice([(0, False), (0, False), (64, False), (64, True)])
        c = _attn("", path, rng.choice(["f32", "f16", "f16", "q8a", "q8a"]), heads, kv, dim, seqs, hi // 8, hi, lens,
                  rope=rope, gate=gate, split=rng.choice([0, 0, 0, 256]), copies=rng.randint(0, min(8, seqs)))
        while work(c)["bytes"] > MAX_BYTES:
            c["hi"] = c["hi"] * 3 // 4
            c["lo"] = c["hi"] // 8
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Inputs


def _ctx(c):
    """Tokens each sequence holds before the pass."""
    r = random.Random(c["lens"])
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["seqs"])]


def _quantise(x):
    """Q8A codes and scales of x [..., dim] (absmax / 127, half away from zero)."""
    amax = x.abs().amax(-1)
    scale = torch.where(amax == 0, torch.ones_like(amax), amax / 127.0)
    y = x / scale[..., None]
    codes = torch.clamp(torch.sign(y) * torch.floor(y.abs() + 0.5), -127, 127).to(torch.int8)
    return codes, scale


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + 17)


def _attn_inputs(c, seed):
    """Everything the pass reads, from the seed alone: pools, tables, lengths, queries, new tokens, gate."""
    g, ctx = _gen(seed), _ctx(c)
    n, kv, d = c["seqs"], c["kv_heads"], c["dim"]
    need = [(L + c["chunk"] + PAGE - 1) // PAGE for L in ctx]
    num_pages = sum(need) + c["copies"] + 8
    order = torch.randperm(num_pages, generator=g, device=DEV).to(torch.int32)
    tables = torch.full((n, max(need)), -1, dtype=torch.int32, device=DEV)  # -1: no page
    at = 0
    for s, k in enumerate(need):
        tables[s, :k] = order[at:at + k]
        at += k
    shape = (num_pages, PAGE, kv, d)
    if c["pages"] == "q8a":
        k, ks = _quantise(torch.randn(shape, generator=g, device=DEV))
        v, vs = _quantise(torch.randn(shape, generator=g, device=DEV))
        ks, vs = ks.reshape(-1, kv), vs.reshape(-1, kv)
    else:
        t = torch.float32 if c["pages"] == "f32" else torch.float16
        k = torch.randn(shape, generator=g, device=DEV, dtype=t)
        v = torch.randn(shape, generator=g, device=DEV, dtype=t)
        ks = vs = None
    rows = n * c["chunk"]
    rand = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x = {"k": k, "v": v, "ks": ks, "vs": vs, "tables": tables, "ctx": ctx, "num_pages": num_pages,
         "q": 2.0 * rand(rows, c["heads"], d), "k_new": rand(rows, kv, d), "v_new": rand(rows, kv, d),
         "gate": torch.sigmoid(rand(rows, c["heads"], d)) if c["gate"] else None}
    # the forked sequences' tail pages: copied from the parents' tails before the step
    x["src"] = torch.stack([tables[s, ctx[s] // PAGE] for s in range(c["copies"])]) if c["copies"] else None
    x["dst"] = order[at:at + c["copies"]].clone() if c["copies"] else None
    return x


def _o_proj_inputs(c, seed):
    r = np.random.default_rng(int(seed) + 5)
    n = c["rows"] * (c["cols"] // 256)
    disk = r.integers(0, 256, (n, 134), dtype=np.uint8)
    disk[:, 0:2] = np.exp2(r.uniform(-9, -5, n)).astype(np.float16).view(np.uint8).reshape(n, 2)
    g = _gen(seed)
    return {"disk": disk, "x": torch.randn((c["vecs"], c["cols"]), generator=g, device=DEV),
            "y": torch.randn((c["vecs"], c["rows"]), generator=g, device=DEV)}


def prepare(case, seed):
    if case["path"] == "o_proj":
        x = _o_proj_inputs(case, seed)
        w = Q4LMatrix(x["disk"], case["rows"], case["cols"], DEV)
        ws = torch.zeros(max(16, w.workspace_size(case["vecs"])), dtype=torch.uint8, device=DEV)
        return {"case": case, "w": w, "x": x["x"], "y": x["y"], "ws": ws}
    c, x = case, _attn_inputs(case, seed)
    pk = PagedKV(x["num_pages"], c["kv_heads"], c["dim"], DTYPES[c["pages"]], DEV)
    for name in ("k", "v", "ks", "vs"):
        if x[name] is not None:
            getattr(pk, name).copy_(x[name])
    s = {"case": case, "pk": pk, "tables": x["tables"], "q": x["q"], "k_new": x["k_new"], "v_new": x["v_new"],
         "gate": x["gate"], "src": x["src"], "dst": x["dst"], "scale": 1.0 / math.sqrt(c["dim"]), "ctx": x["ctx"]}
    s["rope"] = RopeTable(c["rope"], THETA, device=DEV) if c["rope"] else None
    s["out"] = torch.empty_like(x["q"])
    n = c["seqs"]
    if c["path"] == "prompt":
        pos = [L + i for L in x["ctx"] for i in range(c["chunk"])]
        seq = [i for i in range(n) for _ in range(c["chunk"])]
        s["tok_pos"] = torch.tensor(pos, dtype=torch.int32, device=DEV)
        s["tok_seq"] = torch.tensor(seq, dtype=torch.int32, device=DEV)
        s["chunks"] = torch.tensor([[i, L, c["chunk"], i * c["chunk"]] for i, L in enumerate(x["ctx"])],
                                   dtype=torch.int32, device=DEV)
        size = pk.rope_append_workspace_size(s["rope"], n * c["chunk"]) if s["rope"] else 0
        s["ws"] = torch.zeros(max(16, size), dtype=torch.uint8, device=DEV)
    else:
        s["kv_len"] = torch.tensor([L + 1 for L in x["ctx"]], dtype=torch.int32, device=DEV)
        s["max_len"] = max(x["ctx"]) + 1
        if s["rope"]:
            size = pk.rope_decode_workspace_size(s["rope"], n, c["heads"], s["max_len"], c["split"])
        else:
            size = pk.workspace_size(n, c["heads"], s["max_len"], c["split"])
        s["ws"] = torch.zeros(max(16, size), dtype=torch.uint8, device=DEV)
    return s


def run(state):
    s, c = state, state["case"]
    if c["path"] == "o_proj":
        return s["w"].gemv_accumulate(s["x"], s["y"], s["ws"])
    pk = s["pk"]
    if c["path"] == "call":
        pk.attention_paged(s["q"], s["k_new"], s["v_new"], s["tables"][0], s["ctx"][0], c["heads"], out=s["out"])
    elif c["path"] == "prompt":
        if s["rope"]:
            pk.rope_append(s["rope"], s["k_new"], s["v_new"], s["tok_seq"], s["tok_pos"], s["tables"],
                           workspace=s["ws"])
        else:
            pk.append(s["k_new"], s["v_new"], s["tok_seq"], s["tok_pos"], s["tables"])
        pk.prefill_attention(s["q"], s["chunks"], s["tables"], n_heads=c["heads"], scale=s["scale"],
                             window=c["window"], out=s["out"])
    else:
        if c["copies"]:
            pk.page_copy(s["src"], s["dst"])
        kw = dict(n_heads=c["heads"], max_kv_len=s["max_len"], scale=s["scale"], split=c["split"],
                  workspace=s["ws"], out=s["out"])
        if c["gate"]:
            pk.gated_append_decode(s["gate"], s["q"], s["k_new"], s["v_new"], s["tables"], s["kv_len"],
                                   rope=s["rope"], **kw)
        elif s["rope"]:
            pk.rope_append_decode(s["rope"], s["q"], s["k_new"], s["v_new"], s["tables"], s["kv_len"], **kw)
        else:
            pk.append_decode(s["q"], s["k_new"], s["v_new"], s["tables"], s["kv_len"], **kw)
    return {"out": s["out"], "k": pk.k, "v": pk.v, "ks": pk.ks, "vs": pk.vs}


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how close two right answers are


def _attended(c):
    """(pairs of a query and a token it attends, distinct tokens read) of one pass."""
    pairs = tokens = 0
    for L in _ctx(c):
        for i in range(c["chunk"]):
            pairs += min(L + i + 1, c["window"] or L + i + 1)
        tokens += min(L + c["chunk"], (c["window"] or L + c["chunk"]) + c["chunk"] - 1)
    return pairs, tokens


def work(case):
    c = case
    if c["path"] == "o_proj":
        w = c["rows"] * c["cols"] // 256 * 144
        return {"bytes": w + 4 * c["vecs"] * (c["cols"] + 2 * c["rows"]), "flops": 2 * c["rows"] * c["cols"] * c["vecs"]}
    pairs, tokens = _attended(c)
    rows = c["seqs"] * c["chunk"]
    token = 2 * c["kv_heads"] * (c["dim"] * ELEM[c["pages"]] + (4 if c["pages"] == "q8a" else 0))
    page = PAGE * token
    total = tokens * token + rows * (2 * c["kv_heads"] * c["dim"] * 4 + token) + \
        rows * c["heads"] * c["dim"] * 4 * (3 if c["gate"] else 2) + 4 * -(-tokens // PAGE) + c["copies"] * 2 * page
    return {"bytes": total, "flops": 4 * pairs * c["heads"] * c["dim"]}


def tolerance(case):
    """Four times the error against 64 bits that the paths show (o_proj 1.5e-7, f32 pages 3e-7; 4e-7 to 1e-6 where
    f16 pairs carry the queries and the weights)."""
    if case["path"] == "o_proj":
        return {"rel": 6e-7}
    return {"rel": 1.2e-6 if case["pages"] == "f32" else 4e-6}


# ---------------------------------------------------------------------------
# The same in 64 bits


def _turn(x, pos, dim):
    """RoPE of the first `dim` elements of x [rows, heads, d] at positions pos [rows]: angles pos * theta^(-2i/dim)
    as f32 products, each value of the turn rounded to f32 (what the new token's stored K is made from)."""
    half = dim // 2
    inv = torch.pow(torch.tensor(THETA, dtype=torch.float64, device=x.device),
                    -2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dim).float()
    ang = (pos.float()[:, None] * inv[None, :]).double()
    c, s = ang.cos().float()[:, None, :], ang.sin().float()[:, None, :]
    a, b = x[..., :half], x[..., half:dim]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., dim:]], -1)


def _stored(x, pages):
    """A new token's row as the page holds it, in f64."""
    if pages == "q8a":
        codes, scale = _quantise(x)
        return codes.double() * scale.double()[..., None]
    return x.double() if pages == "f32" else x.half().double()


def exact(case, seed):
    c = case
    if c["path"] == "o_proj":
        x = _o_proj_inputs(c, seed)
        disk = torch.from_numpy(x["disk"]).to(DEV)
        glob = disk[:, 0:2].contiguous().view(torch.float16).float()
        loc = torch.stack([disk[:, 2:6] & 15, disk[:, 2:6] >> 4], -1).reshape(-1, 8).float()
        scale = (glob * torch.exp2(loc - 7.0)).half().double()
        nib = torch.stack([disk[:, 6:] & 15, disk[:, 6:] >> 4], -1).reshape(-1, 8, 32).to(torch.int64)
        mag = torch.tensor([0.0] + [2.0 ** (m - 5) for m in range(1, 8)], dtype=torch.float64, device=DEV)
        w = (mag[nib & 7] * (1.0 - 2.0 * (nib >> 3)) * scale[..., None]).reshape(c["rows"], c["cols"])
        return x["y"].double() + x["x"].double() @ w.t().contiguous()
    x, n, kv, d, T = _attn_inputs(c, seed), c["seqs"], c["kv_heads"], c["dim"], c["chunk"]
    rep = c["heads"] // kv
    pos = torch.tensor([L + i for L in x["ctx"] for i in range(T)], dtype=torch.int32, device=DEV)
    k_new = _turn(x["k_new"], pos, c["rope"]) if c["rope"] else x["k_new"]
    q = _turn(x["q"], pos, c["rope"]) if c["rope"] and c["path"] == "step" else x["q"]
    k_new, v_new = _stored(k_new, c["pages"]), _stored(x["v_new"], c["pages"])
    out = torch.empty(x["q"].shape, dtype=torch.float64, device=DEV)
    for s, L in enumerate(x["ctx"]):
        pages = x["tables"][s, :(L + PAGE - 1) // PAGE].long()
        rows = (pages[:, None] * PAGE + torch.arange(PAGE, device=DEV)[None, :]).reshape(-1)[:L]
        at = slice(s * T, (s + 1) * T)
        for h in range(kv):
            old = []
            for p, sc in ((x["k"], x["ks"]), (x["v"], x["vs"])):
                t = p.view(-1, kv, d)[rows, h].double()
                old.append(t * sc[rows, h].double()[:, None] if sc is not None else t)
            K = torch.cat([old[0], k_new[at, h]])
            V = torch.cat([old[1], v_new[at, h]])
            score = q[at, h * rep:(h + 1) * rep].double().reshape(T * rep, d) @ K.t().contiguous() / math.sqrt(d)
            if T > 1 or c["window"]:
                i = torch.arange(T, device=DEV).repeat_interleave(rep)[:, None] + L
                j = torch.arange(L + T, device=DEV)[None, :]
                seen = (j <= i) & (j > i - (c["window"] or L + T + 1))
                score = score.masked_fill(~seen, -math.inf)
            out[at, h * rep:(h + 1) * rep] = (torch.softmax(score, -1) @ V).reshape(T, rep, d)
    if c["gate"]:
        out = out * x["gate"].double()
    # the pools hold copies and conversions, not sums: nothing to compute in 64 bits
    return {"out": out, "k": None, "v": None, "ks": None, "vs": None}
