"""The work that a user of this framework has it do, as cases that can be timed.

A case is a dict of plain values; prepare(case, seed) makes on the GPU what a
serving program has in hand before the call (paged K/V caches, the packed and
uploaded plan, activations, a workspace), run(state) makes the calls of one
pass and returns every output, and exact(case, seed) is the same function in
64 bits on plain torch. Sequence lengths are part of a case (drawn from its
"lengths" number), values come from the seed.

The kinds of case ("call"):
  attn       ragged_paged_attention over a packed step
  store      the same with the step's new K/V rows stored in the call
  qkv        ragged_paged_attention_qkv: bias, RoPE, K/V store and attention
             from the stacked projection rows
  qkv_rms    the same with the pre-attention RMSNorm folded in (what the bf16
             engine runs in every layer)
  reference  attention_decode, the reference launcher's arguments
  argmax     argmax_rows over a step's logits
  model      Model.forward, one whole step of the engine's model
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
if str(ROOT / "llm-engine_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "llm-engine_amd"))

from llm_engine_amd import _lib, engine, kernels  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
MAX_POS = 16384
RMS_EPS = 1e-5


def _attention(name, call, heads, decode=0, ctx=(1, 1), log=False, chunks=0, rows=0, hist=(0, 0), act="bf16",
               kv="bf16", block=16, layers=1, lengths=1):
    """decode rows with contexts drawn from ctx (over their logarithm with log), and chunks prefill chunks of
    `rows` query rows after histories drawn from hist."""
    c = dict(call=call, q_heads=heads[0], kv_heads=heads[1], head_dim=heads[2], decode=decode, ctx_lo=ctx[0],
             ctx_hi=ctx[1], log=log, chunks=chunks, rows=rows, hist_lo=hist[0], hist_hi=hist[1], act=act, kv=kv,
             block=block, layers=layers, lengths=lengths)
    if name:
        c["name"] = name
    return c


def listed():
    qwen, llama, wide = (14, 2, 64), (32, 4, 64), (32, 8, 128)  # Qwen2.5-0.5B, TinyLlama-1.1B, a head_dim-128 GQA-4 shape
    return [
        # One user, one sequence: a decode step's layer, where latency and launches count.
        _attention("decode_one", "qkv", qwen, decode=1, ctx=(700, 700)),
        # A running batch: 64 sequences of very different ages, four layers with a pool each.
        _attention("decode_mix", "qkv", qwen, decode=64, ctx=(64, 4096), log=True, layers=4, lengths=2),
        # A full batch of long contexts: the bandwidth end of decode, fp32 activations.
        _attention("decode_long", "attn", qwen, decode=64, ctx=(4096, 4096), act="f32"),
        # The fp32 engine's decode step (exact fp32 keys and values), storing its new rows.
        _attention("decode_f32", "store", qwen, decode=48, ctx=(32, 2048), log=True, act="f32", kv="f32", layers=2,
                   lengths=3),
        # The bf16 engine's decode step at 64 sequences, norm folded in.
        _attention("decode_llama", "qkv_rms", llama, decode=64, ctx=(128, 1280), layers=2, lengths=4),
        # A program that calls the reference launcher's signature, fp16 as the reference, head_dim 128.
        _attention("decode_reference", "reference", wide, decode=24, ctx=(100, 3000), act="f16", kv="f16", lengths=5),
        # Continuous batching: 32 decode rows beside two prefill chunks of 512, one of them after 1024 cached tokens.
        _attention("mixed", "qkv", qwen, decode=32, ctx=(256, 2048), chunks=2, rows=512, hist=(0, 1024), layers=2,
                   lengths=6),
        # Admission of a burst: the scheduler's default budget of 4096 tokens as eight chunks of 512.
        _attention("prefill_batch", "qkv", llama, chunks=8, rows=512, hist=(0, 1536), lengths=7),
        # One long document: a 2048-row chunk after 8192 cached tokens, head_dim 128.
        _attention("prefill_long", "attn", wide, chunks=1, rows=2048, hist=(8192, 8192), lengths=8),
        # The fp32 engine's mixed step at odd sizes.
        _attention("mixed_f32", "store", qwen, decode=5, ctx=(40, 900), chunks=3, rows=333, hist=(0, 700), act="f32",
                   kv="f32", lengths=9),
        # Greedy selection of a 64-sequence step over the largest vocabulary of the configurations.
        dict(name="argmax", call="argmax", rows=64, vocab=151936),
        # A whole decode step of the bf16 engine: TinyLlama's layers (two of them, and a short vocabulary, so that
        # weights are made quickly and the logits' copy to the host does not hide the step).
        dict(name="model_decode", call="model", decode=64, ctx_lo=64, ctx_hi=512, chunks=0, rows=0, layers=2,
             vocab=4096, lengths=10),
    ]


HEADS = [(14, 2, 64), (32, 4, 64), (32, 8, 128), (16, 16, 64), (28, 4, 128), (8, 8, 128)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: 1 to 256 decode rows with contexts of 1 to 8192 keys, chunks of 2 to 2048
    rows after 0 to 8192 cached keys, every cache type, block sizes 8 to 64, argmax over 1 to 64 rows of 1000 to
    151936 logits, model steps of 1 to 64 rows."""
    limit = max(_cost(c) for c in listed())
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "mixed", "mixed", "argmax", "model"])
    if kind == "argmax":
        return dict(call="argmax", rows=_log(rng, 1, 64), vocab=_log(rng, 1000, 151936))
    if kind == "model":
        chunks = rng.choice([0, 0, 1, 2])
        return dict(call="model", decode=_log(rng, 1, 64), ctx_lo=16, ctx_hi=_log(rng, 32, 512), chunks=chunks,
                    rows=_log(rng, 16, 256) if chunks else 0, layers=2, vocab=4096, lengths=rng.randrange(1 << 20))
    heads = rng.choice(HEADS)
    kv = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    act = rng.choice([kv, kv, "f32"])
    block = rng.choice([16, 16, 16, 8, 32, 64])
    lengths = rng.randrange(1 << 20)
    for _ in range(64):
        if kind == "decode":
            hi = _log(rng, 32, 8192)
            c = _attention(None, rng.choice(["attn", "store", "qkv", "qkv", "qkv_rms", "reference"]), heads,
                           decode=_log(rng, 1, 256), ctx=(rng.choice([1, max(1, hi // 8), hi]), hi),
                           log=rng.random() < 0.5, act=act, kv=kv, block=block, layers=rng.choice([1, 2]),
                           lengths=lengths)
        else:
            hist = rng.choice([0, _log(rng, 16, 8192)])
            c = _attention(None, rng.choice(["attn", "store", "qkv", "qkv_rms"]), heads,
                           decode=_log(rng, 1, 64) if kind == "mixed" else 0, ctx=(16, _log(rng, 32, 4096)),
                           chunks=_log(rng, 1, 8), rows=_log(rng, 2, 2048), hist=(hist // 2, hist), act=act, kv=kv,
                           block=block, lengths=lengths)
        n = c["chunks"] * c["rows"]
        # a step's budget, and the workspace's arrival counters (one per row and kv head, 65536 at most)
        fits = n <= 4096 and (n + c["decode"]) * heads[1] <= 65536
        if fits and _cost(c) <= limit and _output_bytes(c) <= 256 << 20:
            return c
    return _attention(None, "qkv", heads, decode=7, ctx=(33, 777), act=act, kv=kv, block=block, lengths=lengths)


def _output_bytes(c):
    """Bytes of the caches that a case returns (those that its call writes)."""
    if c["call"] in ("attn", "reference"):
        return 0
    start, rows = _spans(c)
    return int((start + rows).sum()) * c["kv_heads"] * c["head_dim"] * 2 * SIZE[c["kv"]] * c["layers"]


def _cost(c):
    """A rough time of one pass, to keep drawn cases below the largest listed one."""
    w = work(c)
    return w["bytes"] / 2e12 + w["flops"] / (0.15e15 if c.get("kv", "bf16") != "f32" else 0.03e15)


# ---- sequence lengths: part of the case ----
def _spans(c):
    """First position and row count of every sequence of the step, prefill chunks first as the scheduler orders them."""
    rng = np.random.default_rng(c["lengths"])
    start, rows = [], []
    for _ in range(c["chunks"]):
        start.append(int(rng.integers(c.get("hist_lo", 0), c.get("hist_hi", 0) + 1)))
        rows.append(c["rows"])
    for _ in range(c["decode"]):
        lo, hi = c["ctx_lo"], c["ctx_hi"]
        n = round(math.exp(rng.uniform(math.log(lo), math.log(hi)))) if c.get("log") else rng.integers(lo, hi + 1)
        start.append(int(n) - 1)
        rows.append(1)
    return np.array(start, dtype=np.int64), np.array(rows, dtype=np.int64)


def work(case):
    c = case
    if c["call"] == "argmax":
        return {"bytes": c["rows"] * (c["vocab"] * 4 + 4), "flops": 0}
    start, rows = _spans(c)
    n, keys = int(rows.sum()), int((start + rows).sum())
    pairs = int((rows * start + rows * (rows + 1) // 2).sum())  # (query, key) pairs under the causal mask
    if c["call"] == "model":
        a = _arch(c)
        kvd, qd = a["kv_heads"] * a["head_dim"], a["q_heads"] * a["head_dim"]
        params = (2 * qd + 2 * kvd + 3 * a["inter"]) * a["hidden"] * a["layers"]
        head = a["vocab"] * a["hidden"]
        return {"bytes": 2 * (params + head) + 4 * keys * kvd * a["layers"] + 4 * len(rows) * a["vocab"],
                "flops": 2 * n * params + 2 * len(rows) * head + 4 * qd * pairs * a["layers"]}
    qd, kvd = c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    act, kv = SIZE[c["act"]], SIZE[c["kv"]]
    layer = keys * kvd * 2 * kv + 2 * n * qd * act + int(((start + rows + c["block"] - 1) // c["block"]).sum()) * 4
    if c["call"] in ("store", "qkv", "qkv_rms"):
        layer += n * kvd * 2 * (act + kv)  # the new rows: read, and written to the cache
    if c["call"] == "qkv_rms":
        layer += n * _hidden(c) * act
    return {"bytes": layer * c["layers"], "flops": 4 * qd * pairs * c["layers"]}


def tolerance(case):
    if case["call"] == "argmax":
        return "exact"
    if case["call"] == "model":  # two bf16 layers: 9e-3 measured
        return {"rel": 3e-2, "max": 0.3}
    if case["kv"] == "f32":
        # sums of fp32 products (4e-7 measured against 64 bits)
        return {"rel": 4e-6}
    # q and the softmax weights in 16 bits (fp16 2.5e-4 to 4e-4, bf16 3.3e-3 measured)
    return {"rel": 1.2e-3 if case["kv"] == "f16" and case["act"] != "bf16" else 1.2e-2}


# ---- attention cases ----
def _hidden(c):
    return c["q_heads"] * c["head_dim"]


def _inputs(c, seed):
    """Device tensors of an attention case, layer by layer, and its block tables."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    start, rows = _spans(c)
    n, hd = int(rows.sum()), c["head_dim"]
    qd, kvd = c["q_heads"] * hd, c["kv_heads"] * hd
    blocks = (start + rows + c["block"] - 1) // c["block"]
    pool = int(blocks.sum()) + 16
    perm = np.random.default_rng(seed).permutation(pool).astype(np.int32)  # a pool in use: no two neighbours in order
    tables = np.split(perm[:int(blocks.sum())], np.cumsum(blocks)[:-1])
    act, kv = DTYPES[c["act"]], DTYPES[c["kv"]]

    def normal(*shape, dtype):
        return torch.randn(*shape, device=dev, generator=g).to(dtype)

    layers = []
    for _ in range(c["layers"]):
        L = dict(k=normal(pool * c["block"], kvd, dtype=kv), v=normal(pool * c["block"], kvd, dtype=kv))
        if c["call"] in ("qkv", "qkv_rms"):
            L["qkv"] = normal(n, qd + 2 * kvd, dtype=act)
            L["bias"] = 0.5 * normal(qd + 2 * kvd, dtype=torch.float32) if c["call"] == "qkv" else None
            L["x"] = 1.5 * normal(n, _hidden(c), dtype=act) if c["call"] == "qkv_rms" else None
        else:
            L["q"] = normal(n, qd, dtype=act)
            if c["call"] == "store":
                L["k_new"], L["v_new"] = normal(n, kvd, dtype=act), normal(n, kvd, dtype=act)
        layers.append(L)
    return dev, start, rows, tables, layers


def _rope(c, dev):
    inv = 1e6 ** (-torch.arange(0, c["head_dim"], 2, device=dev, dtype=torch.float64) / c["head_dim"])
    ang = torch.arange(MAX_POS, device=dev, dtype=torch.float64)[:, None] * inv
    return ang.cos().float(), ang.sin().float()


def _prepare_attention(c, seed):
    dev, start, rows, tables, layers = _inputs(c, seed)
    n, hd = int(rows.sum()), c["head_dim"]
    act = DTYPES[c["act"]]
    s = dict(case=c, layers=layers, scale=1.0 / math.sqrt(hd), stream=torch.cuda.current_stream())
    for L in layers:
        L["out"] = torch.empty(n, c["q_heads"] * hd, device=dev, dtype=act)
    if c["call"] == "reference":
        seq = np.repeat(np.arange(len(rows), dtype=np.int32), rows)
        pos = np.concatenate([np.arange(a, a + r, dtype=np.int32) for a, r in zip(start, rows)])
        off = np.concatenate([[0], np.cumsum([len(t) for t in tables])[:-1]]).astype(np.int32)
        s["index"] = [torch.from_numpy(a).to(dev) for a in (np.concatenate(tables), off, seq, pos)]
        s["ws"] = kernels.new_workspace(kernels.attention_decode_workspace_size(n, c["q_heads"], c["kv_heads"], hd), dev)
        return s
    slices = [kernels.Slice(i, int(start[i]), int(rows[i]), True, tables[i],
                            np.zeros(int(start[i] + rows[i]), dtype=np.int32)) for i in range(len(rows))]
    s["plan"] = kernels.Plan(slices, c["q_heads"], c["kv_heads"], hd, c["block"], DTYPES[c["kv"]],
                             flags=_lib.LE_PLAN_XCD_LOCAL).upload()
    s["ws"] = kernels.new_workspace(s["plan"].workspace_size(), dev)
    if c["call"] in ("qkv", "qkv_rms"):
        s["cos"], s["sin"] = _rope(c, dev)
        s["q_scratch"] = torch.empty(n, c["q_heads"] * hd, device=dev, dtype=act)
    return s


def _run_attention(s):
    c, outs = s["case"], []
    for L in s["layers"]:
        if c["call"] in ("qkv", "qkv_rms"):
            kernels.ragged_paged_attention_qkv(L["qkv"], L["bias"], s["cos"], s["sin"], L["k"], L["v"], s["plan"],
                                               s["scale"], out=L["out"], workspace=s["ws"], q_scratch=s["q_scratch"],
                                               rms_x=L["x"], rms_eps=RMS_EPS)
        elif c["call"] == "store":
            kernels.ragged_paged_attention(L["q"], L["k"], L["v"], s["plan"], s["scale"], out=L["out"],
                                           workspace=s["ws"], k_new=L["k_new"], v_new=L["v_new"])
        elif c["call"] == "attn":
            kernels.ragged_paged_attention(L["q"], L["k"], L["v"], s["plan"], s["scale"], out=L["out"],
                                           workspace=s["ws"])
        else:
            kernels.attention_decode(L["q"], L["k"], L["v"], *s["index"], c["q_heads"], c["kv_heads"], c["head_dim"],
                                     c["block"], s["scale"], out=L["out"], workspace=s["ws"])
        outs.append(L["out"])
        if c["call"] not in ("attn", "reference"):
            outs += [L["k"], L["v"]]
    return outs


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    cos, sin = cos[:, None], sin[:, None]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _causal_attention(q, k, v, first, scale):
    """Rows q [T, H, d] at positions first.. over keys k, v [C, KH, d], in 64 bits."""
    T, H, d = q.shape
    C, KH = k.shape[:2]
    o = torch.empty_like(q)
    mask = torch.arange(C, device=q.device)[None] > torch.arange(first, first + T, device=q.device)[:, None]
    for h in range(H):
        j = h // (H // KH)
        w = (q[:, h] @ k[:, j].T.contiguous()) * scale
        o[:, h] = torch.softmax(w.masked_fill_(mask, -math.inf), dim=-1) @ v[:, j]
    return o


def _exact_attention(c, seed):
    dev, start, rows, tables, layers = _inputs(c, seed)
    H, KH, hd, bs = c["q_heads"], c["kv_heads"], c["head_dim"], c["block"]
    pos = torch.cat([torch.arange(a, a + r, device=dev) for a, r in zip(start.tolist(), rows.tolist())])
    flat = [torch.from_numpy(t).to(dev).long() for t in tables]
    at = [(t[:, None] * bs + torch.arange(bs, device=dev)).reshape(-1) for t in flat]
    slots = torch.cat([s[a:a + r] for s, a, r in zip(at, start.tolist(), rows.tolist())])
    outs = []
    for L in layers:
        k, v = L["k"].double(), L["v"].double()
        if c["call"] in ("qkv", "qkv_rms"):
            x = L["qkv"].double()
            if L["x"] is not None:
                x = x / (L["x"].double().square().mean(-1, keepdim=True) + RMS_EPS).sqrt()
            if L["bias"] is not None:
                x = x + L["bias"].double()
            cos, sin = (t[pos].double() for t in _rope(c, dev))
            q, kn, vn = x.split([H * hd, KH * hd, KH * hd], dim=-1)
            q = _rotate(q.reshape(-1, H, hd), cos, sin)
            k[slots], v[slots] = _rotate(kn.reshape(-1, KH, hd), cos, sin).reshape(-1, KH * hd), vn
        else:
            q = L["q"].double().reshape(-1, H, hd)
            if c["call"] == "store":
                k[slots], v[slots] = L["k_new"].double(), L["v_new"].double()
        o, r0 = [], 0
        for s, a, r in zip(at, start.tolist(), rows.tolist()):
            kk, vv = (t[s[:a + r]].reshape(-1, KH, hd) for t in (k, v))
            o.append(_causal_attention(q[r0:r0 + r], kk, vv, a, 1.0 / math.sqrt(hd)))
            r0 += r
        outs.append(torch.cat(o).reshape(-1, H * hd))
        if c["call"] not in ("attn", "reference"):
            outs += [k, v]
    return outs


# ---- greedy selection ----
def _logits(c, seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    return torch.randn(c["rows"], c["vocab"], device="cuda:0", generator=g) * 3


# ---- the model ----
def _arch(c):
    return dict(engine.ARCHS["tinyllama-1.1b"], layers=c["layers"], vocab=c["vocab"])


def _weights(c, seed):
    a, rng = _arch(c), np.random.default_rng(seed)
    H, I, V = a["hidden"], a["inter"], a["vocab"]
    qd, kvd = a["q_heads"] * a["head_dim"], a["kv_heads"] * a["head_dim"]

    def normal(*shape):
        x = rng.standard_normal(shape, dtype=np.float32)
        x *= np.float32(0.02)
        return x

    def norm():
        return rng.uniform(0.5, 1.5, H).astype(np.float32)

    w = engine.Weights(a, normal(V, H) * np.float32(10), norm(), normal(V, H))
    for _ in range(a["layers"]):
        w.layers.append(dict(wq=normal(qd, H), wk=normal(kvd, H), wv=normal(kvd, H), wo=normal(H, qd),
                             wgate=normal(I, H), wup=normal(I, H), wdown=normal(H, I), in_norm=norm(),
                             post_norm=norm()))
    start, rows = _spans(c)
    tokens = [rng.integers(0, V, int(a + r)).astype(np.int32) for a, r in zip(start, rows)]
    return w, start, rows, tokens


def _prepare_model(c, seed):
    w, start, rows, tokens = _weights(c, seed)
    blocks = (start + rows + 15) // 16
    pool = int(blocks.sum()) + 16
    perm = np.random.default_rng(seed).permutation(pool).astype(np.int32)
    tables = [np.ascontiguousarray(t) for t in np.split(perm[:int(blocks.sum())], np.cumsum(blocks)[:-1])]
    model = engine.Model(w, pool, 16, dtype="bf16")

    def step(items):
        return (_lib.StepSlice * len(items))(*[
            _lib.StepSlice(i, a, n, int(last), tables[i].size, tables[i].ctypes.data, tokens[i].ctypes.data)
            for i, a, n, last in items])

    for i, a in enumerate(start.tolist()):  # the history, chunk by chunk
        for b in range(0, a, 512):
            model.forward(step([(i, b, min(512, a - b), False)]), 0)
    slices = step([(i, int(start[i]), int(rows[i]), True) for i in range(len(rows))])
    return dict(case=c, model=model, slices=slices, n=len(rows), keep=(tables, tokens))


def _exact_model(c, seed):
    """The whole forward of every sequence in 64 bits (RMSNorm, rotate_half RoPE, GQA attention, SwiGLU)."""
    w, start, rows, tokens = _weights(c, seed)
    a, dev = w.arch, torch.device("cuda:0")

    def d(x):
        return torch.from_numpy(x).to(dev).double()

    def norm(x, g):
        return x / (x.square().mean(-1, keepdim=True) + a["eps"]).sqrt() * d(g)

    H, KH, hd = a["q_heads"], a["kv_heads"], a["head_dim"]
    inv = a["theta"] ** (-torch.arange(0, hd, 2, device=dev, dtype=torch.float64) / hd)
    x = d(w.embed)[torch.from_numpy(np.concatenate(tokens)).to(dev).long()]
    n = [len(t) for t in tokens]
    ang = torch.cat([torch.arange(m, device=dev, dtype=torch.float64) for m in n])[:, None] * inv
    for L in w.layers:
        y = norm(x, L["in_norm"])
        q, k = (_rotate((y @ d(L[m]).T).reshape(-1, h, hd), ang.cos(), ang.sin()) for m, h in (("wq", H), ("wk", KH)))
        v = (y @ d(L["wv"]).T).reshape(-1, KH, hd)
        o = torch.cat([_causal_attention(*p, 0, 1.0 / math.sqrt(hd)) for p in zip(q.split(n), k.split(n), v.split(n))])
        x = x + o.reshape(-1, H * hd) @ d(L["wo"]).T
        y = norm(x, L["post_norm"])
        x = x + (torch.nn.functional.silu(y @ d(L["wgate"]).T) * (y @ d(L["wup"]).T)) @ d(L["wdown"]).T
    last = torch.tensor(np.cumsum(n) - 1, device=dev)
    return norm(x[last], w.final_norm) @ d(w.lm_head).T


# ---- the interface ----
def prepare(case, seed):
    if case["call"] == "argmax":
        return dict(case=case, logits=_logits(case, seed))
    return _prepare_model(case, seed) if case["call"] == "model" else _prepare_attention(case, seed)


def run(state):
    call = state["case"]["call"]
    if call == "argmax":
        return kernels.argmax_rows(state["logits"])
    if call == "model":
        return state["model"].forward(state["slices"], state["n"], want_logits=True)[1]
    return _run_attention(state)


def exact(case, seed):
    if case["call"] == "argmax":
        return None
    return _exact_model(case, seed) if case["call"] == "model" else _exact_attention(case, seed)
