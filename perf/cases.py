"""The work whose speed counts here: one layer's attention over the paged KV
cache (decode and prefill, every cache type), an attention layer of a mixed
serving step, an MLP, whole forward passes of the engine, and the cache
mirror's write and read.  Sizes are those of bench.py's configurations (14 / 2
heads x 64 and 32 / 8 heads x 128, 24 layers of 896 / 4864, contexts up to
32k) and generic ones (a 4096-wide layer).

A case is a dict of plain values; `kind` names the path, "lens" seeds the
ragged context lengths (they belong to the case, so the work of a case is
fixed), "q" and "past" list the new and the cached tokens of each prefill
sequence, and the tensors' values come from the seed given to prepare.
"""
import importlib.util
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda:0"
BS = 16  # tokens per cache block
LARGE = {"heads": 32, "kv_heads": 8, "head_dim": 128}
SMALL = {"heads": 14, "kv_heads": 2, "head_dim": 64}
VOCAB = 151936


def package():
    """The vllm-lite_amd directory as the package vllm_lite_amd."""
    if "vllm_lite_amd" not in sys.modules:
        where = os.path.join(ROOT, "vllm-lite_amd")
        spec = importlib.util.spec_from_file_location(
            "vllm_lite_amd", os.path.join(where, "__init__.py"),
            submodule_search_locations=[where])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vllm_lite_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["vllm_lite_amd"]


def listed():
    return [
        # The smallest calls: a few short f32 contexts (the reference's own
        # data type), where latency and launches count.
        dict(name="decode_f32_small", kind="decode", dtype="f32", batch=8, lo=128, hi=1024,
             shared=0, lens=0, **SMALL),
        # The ordinary decode step of a busy server: 64 sequences at 4k.
        dict(name="decode_4k", kind="decode", dtype="bf16", batch=64, lo=4096, hi=4096,
             shared=0, lens=1, **LARGE),
        # Few long, ragged contexts that share a 4096-token system prompt.
        dict(name="decode_long_shared", kind="decode", dtype="bf16", batch=16, lo=8192,
             hi=32768, shared=4096, lens=3, **LARGE),
        # A half-filled batch of ragged contexts over an FP8 cache.
        dict(name="decode_fp8_ragged", kind="decode", dtype="fp8", batch=37, lo=500, hi=8000,
             shared=0, lens=4, **LARGE),
        # Chunked prefill at its largest: four 2048-token chunks.
        dict(name="prefill_chunks", kind="prefill", dtype="bf16", q="2048 2048 2048 2048",
             past="0 512 1024 2048", **LARGE),
        # Ragged continuation chunks over an FP8 cache.
        dict(name="prefill_fp8_ragged", kind="prefill", dtype="fp8", q="701 123 411",
             past="3001 0 517", **LARGE),
        # Prompts in f32, the reference's own data type.
        dict(name="prefill_f32", kind="prefill", dtype="f32", q="511 129 300 64",
             past="0 256 0 33", **SMALL),
        # One attention layer of a serving step that mixes a prompt chunk with
        # decodes (QKV projection, RoPE, cache write, attention, O projection).
        dict(name="layer_mixed", kind="layer", q="512 77", past="1024 0", decodes=29, lo=100,
             hi=3000, lens=5, **LARGE),
        # The MLP over one request's prompt.
        dict(name="mlp_prompt", kind="mlp", rows=333, hidden=896, inter=4864, norm="rms"),
        # The engine's first step over 32 requests' prompts.
        dict(name="engine_prompts", kind="engine", stage="prompts", requests=32, lo=64, hi=512,
             layers=24, hidden=896, inter=4864, lens=5, **SMALL),
        # The engine's decode step for 32 requests, replayed as it captures it.
        dict(name="engine_decode", kind="engine", stage="decode", requests=32, lo=192, hi=640,
             layers=24, hidden=896, inter=4864, lens=6, **SMALL),
        # The reference's cache object: a prompt's K / V written through host
        # index lists and read back.
        dict(name="cache_mirror", kind="mirror", dtype="f32", tokens=1000, kv_heads=2,
             head_dim=64, lens=7),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _text(xs):
    return " ".join(str(x) for x in xs)


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "layer", "mlp", "engine",
                       "mirror"])
    heads = rng.choice([LARGE, SMALL])
    lens = rng.randrange(1 << 20)
    if kind == "decode":
        dtype = rng.choice(["bf16", "bf16", "fp8", "f32"])
        hi = _log_int(rng, 16, 2048 if dtype == "f32" else 32768)
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        batch = _log_int(rng, 1, max(1, min(64, 262144 // hi)))
        shared = 0
        if rng.random() < 0.25 and lo >= 64:
            shared = (lo // 2) // BS * BS
        return dict(kind=kind, dtype=dtype, batch=batch, lo=lo, hi=hi, shared=shared, lens=lens,
                    **heads)
    if kind == "prefill":
        dtype = rng.choice(["bf16", "bf16", "fp8", "f32"])
        if dtype == "f32":
            heads = SMALL
        n = rng.randint(1, 4)
        most = 512 if dtype == "f32" else 2048
        return dict(kind=kind, dtype=dtype, q=_text(_log_int(rng, 16, most) for _ in range(n)),
                    past=_text(rng.choice([0, _log_int(rng, 1, most)]) for _ in range(n)),
                    **heads)
    if kind == "layer":
        n = rng.randint(0, 2)
        return dict(kind=kind, q=_text(_log_int(rng, 16, 1024) for _ in range(n)),
                    past=_text(rng.choice([0, _log_int(rng, 1, 2048)]) for _ in range(n)),
                    decodes=_log_int(rng, 1, 48), lo=_log_int(rng, 16, 500), hi=3000, lens=lens,
                    **heads)
    if kind == "mlp":
        hidden, inter = rng.choice([(896, 4864), (896, 4864), (4096, 12288)])
        return dict(kind=kind, rows=_log_int(rng, 1, 2048 if hidden > 896 else 8192),
                    hidden=hidden, inter=inter, norm=rng.choice(["rms", "rms", "layer"]))
    if kind == "engine":
        stage = rng.choice(["prompts", "decode"])
        return dict(kind=kind, stage=stage, requests=_log_int(rng, 1, 32),
                    lo=_log_int(rng, 16, 64), hi=_log_int(rng, 64, 512), layers=24, hidden=896,
                    inter=4864, lens=lens, **SMALL)
    return dict(kind=kind, dtype=rng.choice(["f32", "bf16"]), tokens=_log_int(rng, 1, 2000),
                kv_heads=heads["kv_heads"], head_dim=heads["head_dim"], lens=lens)


# --- lengths and block tables (of the case alone) ---------------------------

def _contexts(case, count):
    """`count` context lengths, log-uniform in [lo, hi]."""
    rng = random.Random(case["lens"])
    return [_log_int(rng, case["lo"], max(case["lo"], case["hi"])) for _ in range(count)]


def _lengths(case):
    """(new tokens, cached tokens) of each sequence of a prefill / layer case."""
    q, past = ([int(x) for x in case[name].split()] for name in ("q", "past"))
    if case["kind"] == "layer":
        ctx = _contexts(case, case["decodes"])
        q += [1] * len(ctx)
        past += [c - 1 if c > 1 else 1 for c in ctx]
    return q, past


def _blocks(n):
    return (n + BS - 1) // BS


def _tables(lengths, gen, shared=0):
    """Per-sequence block ids, a random permutation of the pool; the first
    shared / 16 blocks are every sequence's.  Returns (lists, pool size)."""
    ns = shared // BS
    pool = ns + sum(_blocks(n) - ns for n in lengths)
    perm = torch.randperm(pool, generator=gen).tolist()
    out, o = [], ns
    for n in lengths:
        k = _blocks(n) - ns
        out.append(perm[:ns] + perm[o:o + k])
        o += k
    return out, pool


def _table_tensor(ids, width=None):
    width = width or max(len(x) for x in ids)
    return torch.tensor([x + [0] * (width - len(x)) for x in ids], dtype=torch.int32)


# --- values (of the seed) ----------------------------------------------------

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.host = torch.Generator().manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.bfloat16):
        return (torch.randn(*shape, generator=self.g, device=DEV) * scale).to(dtype)

    def fp8(self, *shape, scale=0.5):
        """E4M3 codes of normal values (below 2**-6 zero, as the cache's
        encoder flushes them)."""
        x = torch.randn(*shape, generator=self.g, device=DEV) * scale
        code = x.to(torch.float8_e4m3fn).view(torch.uint8)
        return torch.where(x.abs() < 2.0 ** -6, torch.zeros_like(code), code)


def _dt(case):
    return torch.float32 if case["dtype"] == "f32" else torch.bfloat16


def _cache_values(case, r, pool):
    """K [NB, Hkv, 16, D] and V [NB, Hkv, D, 16]."""
    k_shape = (pool, case["kv_heads"], BS, case["head_dim"])
    v_shape = (pool, case["kv_heads"], case["head_dim"], BS)
    if case.get("dtype") == "fp8":
        return r.fp8(*k_shape), r.fp8(*v_shape)
    dt = _dt(case) if "dtype" in case else torch.bfloat16
    return r.normal(*k_shape, scale=0.5, dtype=dt), r.normal(*v_shape, scale=0.5, dtype=dt)


def _attention_values(case, seed):
    """Inputs of a decode or prefill case."""
    r = _Rand(seed)
    if case["kind"] == "decode":
        ctx = _contexts(case, case["batch"])
        rows, q_lens, past = case["batch"], [1] * case["batch"], [c - 1 for c in ctx]
    else:
        q_lens, past = _lengths(case)
        ctx, rows = [a + b for a, b in zip(q_lens, past)], sum(q_lens)
    ids, pool = _tables(ctx, r.host, case.get("shared", 0))
    k, v = _cache_values(case, r, pool)
    q = r.normal(rows, case["heads"], case["head_dim"], dtype=_dt(case))
    return {"ctx": ctx, "q_lens": q_lens, "past": past, "ids": ids, "k": k, "v": v, "q": q}


def _layer_values(case, seed):
    r = _Rand(seed)
    q_lens, past = _lengths(case)
    ids, pool = _tables([a + b for a, b in zip(q_lens, past)], r.host)
    k, v = _cache_values(case, r, pool)
    hq, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    hidden, rows = hq * d, (hq + 2 * hkv) * d
    return {"q_lens": q_lens, "past": past, "ids": ids, "pool": pool, "k": k, "v": v,
            "x": r.normal(sum(q_lens), hidden),
            "wqkv": r.normal(rows, hidden, scale=hidden ** -0.5),
            "bqkv": r.normal(rows, scale=0.1),
            "wo": r.normal(hidden, hidden, scale=hidden ** -0.5)}


def _mlp_values(case, seed):
    r = _Rand(seed)
    h, i = case["hidden"], case["inter"]
    return {"x": r.normal(case["rows"], h), "ln": (1 + r.normal(h, scale=0.1)),
            "wgu": r.normal(2 * i, h, scale=h ** -0.5), "wd": r.normal(h, i, scale=i ** -0.5)}


def _engine_values(case, seed):
    r = _Rand(seed)
    h, i, n, d = case["hidden"], case["inter"], case["layers"], case["head_dim"]
    qkv = (case["heads"] + 2 * case["kv_heads"]) * d
    ones = torch.ones(h, dtype=torch.bfloat16, device=DEV)
    w = {"embed": r.normal(VOCAB, h, scale=0.02), "norm": ones, "ln1": [ones] * n,
         "ln2": [ones] * n,
         "wqkv": [r.normal(qkv, h, scale=0.02) for _ in range(n)],
         "bqkv": [r.normal(qkv, scale=0.02) for _ in range(n)],
         "wo": [r.normal(h, case["heads"] * d, scale=0.02) for _ in range(n)],
         "wgu": [r.normal(2 * i, h, scale=0.02) for _ in range(n)],
         "wd": [r.normal(h, i, scale=0.02) for _ in range(n)]}
    lens = _contexts(case, case["requests"])
    ids, pool = _tables([x + 1 for x in lens], r.host)
    decode = case["stage"] == "decode"
    q_lens, past = ([1] * len(lens), lens) if decode else (lens, [0] * len(lens))
    caches = []
    for _ in range(n):
        shape = (pool, case["kv_heads"], BS, d)
        k, v = r.normal(*shape, scale=0.5), r.normal(shape[0], shape[1], d, BS, scale=0.5)
        caches.append((k, v) if decode else (torch.zeros_like(k), torch.zeros_like(v)))
    tokens = torch.randint(0, VOCAB, (sum(q_lens),), generator=r.host).to(DEV)
    return {"w": w, "q_lens": q_lens, "past": past, "ids": ids, "pool": pool, "caches": caches,
            "tokens": tokens}


def _mirror_values(case, seed):
    r = _Rand(seed)
    shape = (case["tokens"], case["kv_heads"], case["head_dim"])
    ids, pool = _tables([case["tokens"]], r.host)
    return {"k": r.normal(*shape, dtype=_dt(case)), "v": r.normal(*shape, dtype=_dt(case)),
            "ids": ids[0], "pool": pool + 16}


# --- the program's side ------------------------------------------------------

def _i32(xs):
    return torch.tensor(xs, dtype=torch.int32, device=DEV)


def _cumulative(xs):
    out = [0]
    for x in xs:
        out.append(out[-1] + x)
    return out


def _layer_views(cache, layer, owner):
    """A layer's K and V as tensors that keep `owner` (whatever holds the
    library's buffers) alive: the views alone would not."""
    views = cache.key_cache(layer), cache.value_cache(layer)
    for t in views:
        t.owner = owner
    return views


def prepare(case, seed):
    pa = package()
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        s = _attention_values(case, seed)
        s["bt"] = _table_tensor(s["ids"]).to(DEV)
        s["out"] = torch.empty_like(s["q"])
        if kind == "decode":
            s["ctx_dev"], s["max_ctx"] = _i32(s["ctx"]), max(s["ctx"])
            size = pa.decode_workspace_size(case["batch"], case["heads"], case["head_dim"],
                                            s["max_ctx"])
            s["ws"] = torch.empty(max(size, 1), dtype=torch.uint8, device=DEV)
        else:
            s["cu"], s["past_dev"] = _i32(_cumulative(s["q_lens"])), _i32(s["past"])
    elif kind == "layer":
        s = _layer_values(case, seed)
        cache = pa.PagedKvCache(1, case["kv_heads"], case["head_dim"], s["pool"],
                                torch.bfloat16, DEV)
        s["cache"] = cache
        s["kc"], s["vc"] = _layer_views(cache, 0, cache)
        s["kc"].copy_(s.pop("k"))
        s["vc"].copy_(s.pop("v"))
        s["inv_freq"] = torch.from_numpy(pa.rope_inv_freq(case["head_dim"], 1e6)).to(DEV)
        s["batch"] = pa.StepBatch()
        s["batch"].prepare(cache, s["q_lens"], s["past"], s["ids"])
    elif kind == "mlp":
        s = _mlp_values(case, seed)
        if case["rows"] <= 64:  # a decode step's weights, packed once
            fold = s["ln"] if case["norm"] == "rms" else None
            s["gu"] = pa.ops.PackedWeight(s["wgu"], col_scale=fold)
            s["down"] = pa.ops.PackedWeight(s["wd"])
            s["ws"] = pa.ops.linear_workspace(case["rows"], case["hidden"], case["inter"])
    elif kind == "engine":
        from vllm_lite_amd import e2e
        s = _engine_values(case, seed)
        cfg = e2e.ModelConfig(layers=case["layers"], hidden=case["hidden"], heads=case["heads"],
                              kv_heads=case["kv_heads"], head_dim=case["head_dim"],
                              inter=case["inter"], vocab=VOCAB)
        w = e2e.Weights(cfg, device=DEV)
        for name, value in s.pop("w").items():
            setattr(w, name, value)
        w.pack()
        eng = e2e.Engine(cfg, w, s["pool"], device=DEV)
        caches = []
        for layer, (k, v) in enumerate(s.pop("caches")):
            kc, vc = _layer_views(eng.cache, layer, eng)
            kc.copy_(k)
            vc.copy_(v)
            caches += [kc, vc]
        s.update(eng=eng, caches=caches)
        if case["stage"] == "prompts":
            s["last"] = torch.tensor([x - 1 for x in _cumulative(s["q_lens"])[1:]], device=DEV)
        else:
            # the decode step captured once, as the engine's own generation does
            eng.batch.set_capacity(max(s["past"]) + 1)
            eng.batch.prepare(eng.cache, s["q_lens"], s["past"], s["ids"])
            eng.forward(s["tokens"], None)
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["logits"] = eng.forward(s["tokens"], None)
    else:
        s = _mirror_values(case, seed)
        s["cache"] = pa.PagedKvCache(1, case["kv_heads"], case["head_dim"], s["pool"],
                                     _dt(case), DEV)
        s["pos"] = list(range(case["tokens"]))
    s["case"], s["pa"] = case, pa
    return s


def run(s):
    case, pa = s["case"], s["pa"]
    kind = case["kind"]
    if kind == "decode":
        return pa.decode(s["q"], s["k"], s["v"], s["bt"], s["ctx_dev"], s["max_ctx"],
                         out=s["out"], workspace=s["ws"])
    if kind == "prefill":
        return pa.prefill(s["q"], s["k"], s["v"], s["bt"], s["cu"], s["past_dev"],
                          max(s["q_lens"]), out=s["out"])
    if kind == "layer":
        hq, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
        t, nq = s["x"].shape[0], hq * d
        qkv = pa.linear(s["x"], s["wqkv"], s["bqkv"])
        q = qkv[:, :nq].view(t, hq, d)
        k = qkv[:, nq:nq + hkv * d].view(t, hkv, d)
        v = qkv[:, nq + hkv * d:].view(t, hkv, d)
        attn = s["batch"].attention(s["cache"], 0, q, k, v, s["inv_freq"])
        return [pa.linear(attn.reshape(t, nq), s["wo"]), s["kc"], s["vc"]]
    if kind == "mlp":
        norm = pa.rms_norm if case["norm"] == "rms" else pa.layer_norm
        swiglu = pa.ops.ACT_SILU_MUL
        if case["rows"] <= 64:
            if case["norm"] == "rms":
                act = pa.linear(s["x"], s["gu"], act=swiglu, rms_eps=1e-6)
            else:
                act = pa.linear(norm(s["x"], s["ln"], 1e-6), s["gu"], act=swiglu)
            return pa.linear(act, s["down"], workspace=s["ws"])
        act = pa.linear(norm(s["x"], s["ln"], 1e-6), s["wgu"], act=swiglu)
        return pa.linear(act, s["wd"])
    if kind == "engine":
        if case["stage"] == "decode":
            s["graph"].replay()
            return [s["logits"]] + s["caches"]
        eng = s["eng"]
        eng.batch.prepare(eng.cache, s["q_lens"], s["past"], s["ids"])
        return [eng.forward(s["tokens"], s["last"])] + s["caches"]
    s["cache"].write_prefill_kv(0, s["ids"], s["pos"], case["tokens"], s["k"], s["v"])
    return list(s["cache"].read_kv(0, s["ids"], case["tokens"]))


# --- what a pass cannot do without --------------------------------------------

def _pairs(q_lens, past):
    """(query, key) pairs under the causal rule."""
    return sum(n * p + n * (n + 1) // 2 for n, p in zip(q_lens, past))


def work(case):
    kind = case["kind"]
    if kind == "mirror":
        return {"bytes": 8 * case["tokens"] * case["kv_heads"] * case["head_dim"] *
                (4 if case["dtype"] == "f32" else 2), "flops": 0}
    if kind == "mlp":
        r, h, i = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 2 * (3 * h * i + 2 * r * h), "flops": 6 * r * h * i}
    hq, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    if kind in ("decode", "prefill"):
        if kind == "decode":
            past = [c - 1 for c in _contexts(case, case["batch"])]
            q_lens = [1] * len(past)
        else:
            q_lens, past = _lengths(case)
        es = {"f32": 4, "bf16": 2, "fp8": 1}[case["dtype"]]
        shared = case.get("shared", 0)
        keys = sum(q_lens) + sum(past) - shared * (len(past) - 1 if shared else 0)
        rows = sum(q_lens) * hq * d * (4 if case["dtype"] == "f32" else 2)
        return {"bytes": 2 * keys * hkv * d * es + 2 * rows,
                "flops": 4 * hq * d * _pairs(q_lens, past)}
    if kind == "layer":
        q_lens, past = _lengths(case)
        hidden, qkv, layers, extra_b, extra_f = hq * d, (hq + 2 * hkv) * d, 1, 0, 0
    else:
        lens = _contexts(case, case["requests"])
        q_lens, past = ([1] * len(lens), lens) if case["stage"] == "decode" else (lens,
                                                                                  [0] * len(lens))
        hidden, qkv, layers = case["hidden"], (hq + 2 * hkv) * d, case["layers"]
        mlp = 3 * hidden * case["inter"]
        n = len(lens)
        extra_b = 2 * (layers * mlp + VOCAB * hidden) + 4 * n * VOCAB
        extra_f = 2 * (layers * sum(q_lens) * mlp + n * VOCAB * hidden)
    t = sum(q_lens)
    weights = hidden * qkv + hq * d * hidden
    kv = 2 * hkv * d * 2
    return {"bytes": layers * (2 * weights + kv * (sum(past) + t)) + 4 * t * hidden + extra_b,
            "flops": layers * (2 * t * weights + 4 * hq * d * _pairs(q_lens, past)) + extra_f}


def tolerance(case):
    kind = case["kind"]
    if kind == "mirror":
        return "exact"
    if kind == "engine":
        # 24 layers of bf16 activations (1.6e-2 to 3.7e-2 from the 64-bit logits)
        return {"rel": 1e-1}
    if kind in ("layer", "mlp"):
        # two or three bf16 roundings in a row (4e-3 from the 64-bit values)
        return {"rel": 1.6e-2}
    if case["dtype"] == "f32":
        # 32-bit sums throughout (1.8e-7)
        return {"rel": 1e-6}
    return {"rel": 1e-2}  # bf16 probabilities and outputs (2.4e-3)


# --- 64-bit values -----------------------------------------------------------

def _f64(t):
    if t.dtype == torch.uint8:
        return t.view(torch.float8_e4m3fn).to(torch.float64)
    return t.to(torch.float64)


def _attend64(q, k, v, ids, q_lens, past):
    """Causal attention of q [T, Hq, D] over the paged K / V, in 64 bits."""
    hq, d = q.shape[1], q.shape[2]
    hkv = k.shape[1]
    g = hq // hkv
    out, row = [], 0
    for n, p, blocks in zip(q_lens, past, ids):
        ctx = p + n
        idx = torch.tensor(blocks[:_blocks(ctx)], device=DEV)
        kk = _f64(k[idx]).transpose(0, 1).reshape(hkv, -1, d)[:, :ctx]
        vv = _f64(v[idx]).permute(1, 0, 3, 2).reshape(hkv, -1, d)[:, :ctx]
        qq = _f64(q[row:row + n]).view(n, hkv, g, d).permute(1, 2, 0, 3)
        heads = []
        for h in range(hkv):
            s = torch.matmul(qq[h].reshape(g * n, d), kk[h].t().contiguous()) / math.sqrt(d)
            if n > 1:
                keys = torch.arange(ctx, device=DEV)
                last = (p + torch.arange(n, device=DEV)).repeat(g)
                s = s.masked_fill(keys[None, :] > last[:, None], -math.inf)
            heads.append(torch.matmul(torch.softmax(s, -1), vv[h]).view(g, n, d))
        out.append(torch.stack(heads).permute(2, 0, 1, 3).reshape(n, hq, d))
        row += n
    return torch.cat(out)


def _attention_layer64(x, wqkv, bqkv, wo, k, v, ids, q_lens, past, case, theta):
    """QKV projection, RoPE, cache write, attention and O projection; k and v
    (64-bit caches) are updated in place."""
    hq, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    qkv = x @ _f64(wqkv).t() + _f64(bqkv)
    t = x.shape[0]
    pos = torch.tensor([p + i for n, p in zip(q_lens, past) for i in range(n)], device=DEV)
    blk = torch.tensor([b[(p + i) // BS] for n, p, b in zip(q_lens, past, ids)
                        for i in range(n)], device=DEV)
    half = d // 2
    freq = theta ** (-2.0 * torch.arange(half, dtype=torch.float64, device=DEV) / d)
    ang = pos.to(torch.float64)[:, None] * freq.float().double()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(y):
        a, b = y[..., :half], y[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    q = rope(qkv[:, :hq * d].view(t, hq, d))
    k[blk, :, pos % BS] = rope(qkv[:, hq * d:(hq + hkv) * d].view(t, hkv, d))
    v[blk, :, :, pos % BS] = qkv[:, (hq + hkv) * d:].view(t, hkv, d)
    return _attend64(q, k, v, ids, q_lens, past).reshape(t, hq * d) @ _f64(wo).t()


def _norm64(x, w, norm):
    if norm == "layer":
        x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * _f64(w)


def _mlp64(h, wgu, wd):
    gate, up = (h @ _f64(wgu).t()).chunk(2, -1)
    return (torch.nn.functional.silu(gate) * up) @ _f64(wd).t()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        s = _attention_values(case, seed)
        return _attend64(s["q"], s["k"], s["v"], s["ids"], s["q_lens"], s["past"])
    if kind == "layer":
        s = _layer_values(case, seed)
        k, v = _f64(s["k"]), _f64(s["v"])
        y = _attention_layer64(_f64(s["x"]), s["wqkv"], s["bqkv"], s["wo"], k, v, s["ids"],
                               s["q_lens"], s["past"], case, 1e6)
        return [y, k, v]
    if kind == "mlp":
        s = _mlp_values(case, seed)
        return _mlp64(_norm64(_f64(s["x"]), s["ln"], case["norm"]), s["wgu"], s["wd"])
    if kind == "engine":
        s = _engine_values(case, seed)
        w = s["w"]
        x = _f64(w["embed"][s["tokens"]])
        caches = []
        for i in range(case["layers"]):
            k, v = (_f64(c) for c in s["caches"][i])
            x = x + _attention_layer64(_norm64(x, w["ln1"][i], "rms"), w["wqkv"][i],
                                       w["bqkv"][i], w["wo"][i], k, v, s["ids"], s["q_lens"],
                                       s["past"], case, 1e6)
            x = x + _mlp64(_norm64(x, w["ln2"][i], "rms"), w["wgu"][i], w["wd"][i])
            caches += [k, v]
        last = torch.tensor([n - 1 for n in _cumulative(s["q_lens"])[1:]], device=DEV)
        return [_norm64(x[last], w["norm"], "rms") @ _f64(w["embed"]).t()] + caches
    s = _mirror_values(case, seed)
    return [_f64(s["k"]), _f64(s["v"])]
