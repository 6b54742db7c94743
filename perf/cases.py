"""Performance cases of the attention layer calls: decode over paged pools (GQA, absorbed MLA, DSA), the verify step of
speculative decoding, prefill, the QKV writer and the DSA indexer, each through the package's public entry points.

A case is a dict of plain values; ``path`` names the call and the other entries its sizes. A batch's lengths are spread
evenly from ``lo`` to ``hi`` (so the work does not depend on the seed) and dealt to its rows at random; pages lie at
random places of the pool, as a serving allocator leaves them after some time. Small decode calls go through the bound
launch (``ops.prepare_*``), as a serving loop of small batches does; the calls without one go through ``ops`` itself.
"""

from __future__ import annotations

import math

import torch

from sglang_neuron_amd import ops

FP8 = torch.float8_e4m3fn
DEV = "cuda"

# head shapes: (query heads, KV heads, head dim)
QWEN3_8B = dict(H=32, G=8, d=128)
QWEN3_06B = dict(H=16, G=8, d=128)
GPT_OSS_SHARE = dict(H=8, G=1, d=64, sinks=True)  # one of eight ranks' heads


def listed():
    return [
        # one chat user of a small model: the shortest call, where launches and latency are everything
        dict(name="decode-b1", path="gqa", B=1, lo=300, hi=300, **QWEN3_06B, P=16, fp8=False, window=0),
        # a full serving batch at 4k context over an FP8 pool: the ordinary throughput step
        dict(name="decode-b64-fp8", path="gqa", B=64, lo=4096, hi=4096, **QWEN3_8B, P=16, fp8=True, window=0),
        # a ragged GPT-OSS batch on one rank's share of the heads: its full-attention layers, sinks and multipliers
        dict(name="decode-oss-full", path="gqa", B=128, lo=2048, hi=8192, **GPT_OSS_SHARE, P=16, fp8=True, window=0),
        # the same batch in the model's sliding-window layers (every other layer)
        dict(name="decode-oss-window", path="gqa", B=128, lo=2048, hi=8192, **GPT_OSS_SHARE, P=16, fp8=True,
             window=128),
        # speculative decoding's verify step: four tokens a row over a ragged batch
        dict(name="verify-s4-fp8", path="gqa_multi", B=16, S=4, lo=1000, hi=8000, **QWEN3_8B, P=16, fp8=True,
             window=0),
        # DeepSeek-V2-Lite decode, ragged, FP8 rows with their scales
        dict(name="mla-b32-fp8", path="mla", B=32, lo=1024, hi=16384, H=16, P=64, fp8=True),
        # the same model over the bf16 rows and 128-token pages it is served with
        dict(name="mla-b32-bf16", path="mla", B=32, lo=1024, hi=16384, H=16, P=128, fp8=False),
        # a GLM DSA decode step after the indexer: 2048 gathered rows of up to 131072
        dict(name="dsa-b16", path="dsa", B=16, spec=1, lo=1000, hi=131072, H=16, P=64, K=2048),
        # the indexer of that step: the new keys stored, every cached key scored, the top 2048 selected
        dict(name="indexer-b16-128k", path="indexer", B=16, lo=131072, hi=131072, H=64, P=64, K=2048),
        # a prefill batch in chunks: four requests, each 2048 tokens after 2048
        dict(name="prefill-4x2048-fp8", path="prefill", R=4, lo=2048, hi=2048, prior_lo=2048, prior_hi=2048,
             **QWEN3_8B, P=16, fp8=True, window=0),
        # a chat turn on a cached conversation: short new prompts after a long prior, bf16 pool
        dict(name="prefill-turn-bf16", path="prefill", R=2, lo=150, hi=251, prior_lo=9000, prior_hi=17000,
             **QWEN3_8B, P=128, fp8=False, window=0),
        # the writer after the QKV projection of a prefill chunk: QK norm, RoPE, FP8 store
        dict(name="qkv-writer-8192", path="qkv", T=8192, **QWEN3_8B, P=16, fp8=True, norm=True),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["gqa", "gqa", "gqa", "gqa_multi", "mla", "mla", "dsa", "indexer", "prefill", "prefill", "qkv"])
    heads = dict(rng.choice([QWEN3_8B, QWEN3_06B, GPT_OSS_SHARE]))
    sinks = bool(heads.get("sinks"))
    P = rng.choice([16, 16, 128])
    fp8 = rng.random() < 0.6 or sinks
    window = 128 if sinks and rng.random() < 0.5 else 0
    if path in ("gqa", "gqa_multi"):
        c = dict(path=path, B=_log_int(rng, 1, 128), **heads, P=P, fp8=fp8, window=window)
        if path == "gqa_multi":
            c["S"] = rng.choice([2, 3, 4, 5, 8])
            c["B"] = _log_int(rng, 1, 32)
        hi = _log_int(rng, 64, 32768)
        while c["B"] * hi * c["G"] * c["d"] * (2 if fp8 else 4) > 520e6 // (1 if path == "gqa" else 4):
            hi = hi * 2 // 3
        c["hi"] = hi
        c["lo"] = max(16, int(hi * rng.uniform(0.1, 1.0)))
        return c
    if path == "mla":
        c = dict(path=path, B=_log_int(rng, 1, 64), H=16, P=rng.choice([64, 128]), fp8=rng.random() < 0.5)
        hi = _log_int(rng, 64, 32768)
        while c["B"] * hi * (580 if c["fp8"] else 1152) > 400e6:
            hi = hi * 2 // 3
        c["hi"] = hi
        c["lo"] = max(16, int(hi * rng.uniform(0.1, 1.0)))
        return c
    if path == "dsa":
        hi = _log_int(rng, 2048, 131072)
        return dict(path=path, B=_log_int(rng, 1, 16), spec=rng.choice([1, 1, 8]), lo=max(64, int(hi * rng.uniform(0.02, 1.0))),
                    hi=hi, H=16, P=64, K=2048)
    if path == "indexer":
        hi = _log_int(rng, 2048, 131072)
        return dict(path=path, B=_log_int(rng, 1, 16), lo=hi, hi=hi, H=64, P=64, K=2048)
    if path == "prefill":
        c = dict(path=path, R=_log_int(rng, 1, 8), hi=_log_int(rng, 16, 4096), **heads, P=P, fp8=fp8, window=window)
        c["prior_hi"] = rng.choice([0, _log_int(rng, 64, 32768), _log_int(rng, 64, 32768)])
        c["prior_lo"] = int(c["prior_hi"] * rng.uniform(0.1, 1.0))
        while c["R"] * c["hi"] * (c["prior_hi"] + c["hi"]) * 4 * c["d"] * c["H"] > 0.4e12 or c["R"] * c["hi"] > 8192:
            c["hi"] = max(16, c["hi"] * 2 // 3)
            c["R"] = max(1, c["R"] - 1)
        c["lo"] = max(8, int(c["hi"] * rng.uniform(0.2, 1.0)))
        return c
    return dict(path=path, T=_log_int(rng, 1, 8192), **heads, P=P, fp8=fp8, norm=not sinks)


# ---- inputs (plain torch, from the seed alone) ----

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _spread(lo, hi, n):
    return [hi if n == 1 else lo + (hi - lo) * i // (n - 1) for i in range(n)]


def _dealt(lens, g):
    """The lengths in random row order, as a list."""
    order = torch.randperm(len(lens), generator=g, device=DEV).tolist()
    return [lens[i] for i in order]


def _normal(shape, g, scale=1.0):
    x = torch.randn(shape, generator=g, device=DEV)
    return (x * scale if scale != 1.0 else x).to(torch.bfloat16)


def _fp8_normal(shape, g, scale):
    """e4m3fn values of N(0, 1) elements at a dequantization scale (a tensor that broadcasts, or a number)."""
    return (torch.randn(shape, generator=g, device=DEV) / scale).clamp_(-448, 448).to(FP8)


def _pages(lens, P, g):
    """(block table [B, width] int32 on the GPU, pool pages): random pages 1 .. n, page 0 reserved, -1 past a row."""
    per = [-(-n // P) for n in lens]
    perm = (torch.randperm(sum(per), generator=g, device=DEV) + 1).to(torch.int32)
    table = torch.full((len(lens), max(per)), -1, dtype=torch.int32, device=DEV)
    off = 0
    for b, n in enumerate(per):
        table[b, :n] = perm[off:off + n]
        off += n
    return table, sum(per) + 1


def _slots(table, rows, pos, P):
    return table[rows, pos // P].to(torch.int64) * P + pos % P


def _mha_pool(c, nb, g):
    shape = (nb, c["G"], c["P"], c["d"])
    if not c["fp8"]:
        return _normal(shape, g), _normal(shape, g), None, None
    # a checkpoint-like dequantization scale per KV head, absmax / 448 of normal tokens
    s = [(4.5 + torch.rand(c["G"], generator=g, device=DEV)) / 448 for _ in range(2)]
    k, v = (_fp8_normal(shape, g, x.reshape(1, -1, 1, 1)) for x in s)
    if c.get("sinks") and c["path"] in ("gqa", "gqa_multi"):  # GPT-OSS decode: the inverted bf16 scale multiplies
        s = [(1.0 / x.to(torch.bfloat16)).float() for x in s]
    return k, v, s[0], s[1]


def _raw(t):
    """A pool's storage as whole numbers (a view), so that what the store wrote is compared exactly."""
    return t.view(torch.uint8 if t.element_size() == 1 else torch.int16)


def _inputs(c, seed):
    g = _gen(seed)
    s = dict(case=c)
    path = c["path"]
    if path in ("gqa", "gqa_multi"):
        B, H, G, d, P = c["B"], c["H"], c["G"], c["d"], c["P"]
        S = c.get("S", 1)
        lens = [max(n, S) for n in _dealt(_spread(c["lo"], c["hi"], B), g)]
        table, nb = _pages(lens, P, g)
        kc, vc, ks, vs = _mha_pool(c, nb, g)
        q, kn, vn = _normal((B, S, H, d), g), _normal((B, S, G, d), g), _normal((B, S, G, d), g)
        lens_d = torch.tensor(lens, dtype=torch.int32, device=DEV)
        rows = torch.arange(B, device=DEV).repeat_interleave(S)
        pos = (lens_d.long()[:, None] - S + torch.arange(S, device=DEV)).reshape(-1)
        slots = _slots(table, rows, pos, P).reshape(B, S)
        sinks = torch.randn(H, generator=g, device=DEV) if c.get("sinks") else None
        s.update(q=q, kn=kn, vn=vn, kc=kc, vc=vc, ks=ks, vs=vs, table=table, lens=lens, lens_d=lens_d, slots=slots,
                 sinks=sinks)
    elif path == "mla":
        B, H, P = c["B"], c["H"], c["P"]
        lens = _dealt(_spread(c["lo"], c["hi"], B), g)
        table, nb = _pages(lens, P, g)
        rows = torch.randn(nb * P, 576, generator=g, device=DEV)
        rows[:, :512] *= 0.5
        if c["fp8"]:
            sc = rows.abs().amax(dim=1) / 448
            cache = (rows / sc[:, None]).clamp_(-448, 448).to(FP8).view(torch.uint8)
        else:
            cache, sc = rows.to(torch.bfloat16), None
        new = torch.cat([_normal((B, 512), g, 0.5), _normal((B, 64), g)], dim=1)
        lens_d = torch.tensor(lens, dtype=torch.int32, device=DEV)
        slots = _slots(table, torch.arange(B, device=DEV), lens_d.long() - 1, P)
        s.update(ql=_normal((B, H, 512), g), qp=_normal((B, H, 64), g), cache=cache, sc=sc, table=table, lens=lens,
                 lens_d=lens_d, new=new, slots=slots)
    elif path == "dsa":
        B, spec, H, P, K = c["B"], c["spec"], c["H"], c["P"], c["K"]
        lens = _dealt(_spread(c["lo"], c["hi"], B), g)
        table, nb = _pages(lens, P, g)
        n = nb * P
        scale = 2.0 ** -6
        cache = torch.empty(n, 640, dtype=torch.uint8, device=DEV)
        cache[:, :128] = _normal((n, 64), g, 1 / scale).view(torch.uint8)
        cache[:, 128:] = _fp8_normal((n, 512), g, scale).view(torch.uint8)
        idx = torch.full((B * spec, K), -1, dtype=torch.int32, device=DEV)
        for b, length in enumerate(lens):
            prior = length - spec
            for j in range(spec):  # the last 128 positions and a draw of the others, in position order
                if prior <= K:
                    sel = torch.arange(prior, device=DEV)
                else:
                    rest = torch.randperm(prior - 128, generator=g, device=DEV)[:K - 128]
                    sel = torch.cat([rest.sort().values, torch.arange(prior - 128, prior, device=DEV)])
                idx[b * spec + j, :sel.numel()] = sel.to(torch.int32)
        T = B * spec
        pos = torch.tensor([n - spec + j for n in lens for j in range(spec)], dtype=torch.int32, device=DEV)
        slots = _slots(table, torch.arange(T, device=DEV) // spec, pos.long(), P)
        s.update(qa=_normal((T, H, 512), g), qp=_normal((T, H, 64), g), cache=cache, scale=scale, idx=idx, table=table,
                 pos=pos, own=_normal((T, 576), g), slots=slots)
    elif path == "indexer":
        B, H, P = c["B"], c["H"], c["P"]
        lens = _dealt(_spread(c["lo"], c["hi"], B), g)
        table, nb = _pages([n + 1 for n in lens], P, g)
        keys = torch.randn(nb, P, 128, generator=g, device=DEV).to(FP8).view(torch.uint8)
        limits = torch.tensor(lens, dtype=torch.int32, device=DEV)
        s.update(q=_normal((B, H, 128), g), w=torch.rand(B, H, generator=g, device=DEV) * H ** -0.5, keys=keys,
                 new=_normal((B, 128), g), slots=_slots(table, torch.arange(B, device=DEV), limits.long(), P),
                 table=table, limits=limits, width=max(lens))
    elif path == "prefill":
        R, H, G, d, P = c["R"], c["H"], c["G"], c["d"], c["P"]
        chunks = _dealt(_spread(c["lo"], c["hi"], R), g)
        priors = _spread(c["prior_lo"], c["prior_hi"], R)
        table, nb = _pages([a + b for a, b in zip(chunks, priors)], P, g)
        kc, vc, ks, vs = _mha_pool(c, nb, g)
        T = sum(chunks)
        start = [0]
        for n in chunks:
            start.append(start[-1] + n)
        rows = torch.cat([torch.full((n,), r, device=DEV) for r, n in enumerate(chunks)])
        pos = torch.cat([torch.arange(p, p + n, device=DEV) for p, n in zip(priors, chunks)])
        sinks = torch.randn(H, generator=g, device=DEV) if c.get("sinks") else None
        s.update(q=_normal((T, H, d), g), kn=_normal((T, G, d), g), vn=_normal((T, G, d), g), kc=kc, vc=vc, ks=ks,
                 vs=vs, table=table, start=start, priors=priors, slots=_slots(table, rows, pos, P), sinks=sinks,
                 start_d=torch.tensor(start, dtype=torch.int32, device=DEV),
                 priors_d=torch.tensor(priors, dtype=torch.int32, device=DEV), longest=max(chunks))
    else:  # qkv
        T, H, G, d, P = c["T"], c["H"], c["G"], c["d"], c["P"]
        table, nb = _pages([T], P, g)
        kc, vc, ks, vs = _mha_pool(c, nb, g)
        pos = torch.arange(T, device=DEV)
        ang = pos.double()[:, None] / (1.0e6 ** (torch.arange(d // 2, dtype=torch.float64, device=DEV) * 2 / d))
        ang = torch.cat([ang, ang], dim=1)
        gamma = [(1.0 + 0.1 * torch.randn(d, generator=g, device=DEV)).to(torch.bfloat16) for _ in range(2)]
        s.update(qkv=_normal((T, (H + 2 * G) * d), g, 2.0), cos=ang.cos().to(torch.bfloat16),
                 sin=ang.sin().to(torch.bfloat16), gamma=gamma if c["norm"] else [None, None], kc=kc, vc=vc, ks=ks,
                 vs=vs, slots=_slots(table, torch.zeros_like(pos), pos, P))
    return s


# ---- the calls ----

def prepare(case, seed):
    s = _inputs(case, seed)
    c = case
    path = c["path"]
    if path == "gqa":
        s["call"] = ops.prepare_paged_decode_gqa(
            s["q"][:, 0], s["kc"], s["vc"], s["table"], s["lens_d"], s["kn"][:, 0], s["vn"][:, 0],
            sm_scale=c["d"] ** -0.5, k_scale=s["ks"], v_scale=s["vs"], sinks=s["sinks"], window=c["window"],
            new_slots=s["slots"].reshape(-1), host_seq_lens=s["lens"],
            scales_multiply=bool(c["fp8"] and c.get("sinks")))
    elif path == "mla":
        s["call"] = ops.prepare_mla_decode(s["ql"], s["qp"], s["cache"], s["sc"], s["table"], s["lens_d"], s["new"],
                                           sm_scale=192 ** -0.5, page_size=c["P"], new_slots=s["slots"],
                                           host_seq_lens=s["lens"])
    elif path == "dsa":
        s["call"] = ops.prepare_mla_decode_sparse(s["qa"], s["qp"], s["cache"], s["scale"], s["idx"], s["table"],
                                                  s["pos"], s["own"], sm_scale=0.0625, page_size=c["P"],
                                                  new_slots=s["slots"], spec=c["spec"])
    return s


def run(s):
    c = s["case"]
    path = c["path"]
    if path == "gqa":
        return {"out": s["call"](), "k": _raw(s["kc"]), "v": _raw(s["vc"])}
    if path == "gqa_multi":
        out = ops.paged_decode_gqa_multi(s["q"], s["kc"], s["vc"], s["table"], s["lens_d"], s["kn"], s["vn"],
                                         sm_scale=c["d"] ** -0.5, new_slots=s["slots"], k_scale=s["ks"],
                                         v_scale=s["vs"], sinks=s["sinks"], window=c["window"],
                                         scales_multiply=bool(c["fp8"] and c.get("sinks")), host_seq_lens=s["lens"])
        return {"out": out, "k": _raw(s["kc"]), "v": _raw(s["vc"])}
    if path == "mla":
        out = s["call"]()
        return {"out": out, "cache": s["cache"] if c["fp8"] else _raw(s["cache"]), "scale": s["sc"]}
    if path == "dsa":
        ctx, lse = s["call"]()
        return {"out": ctx, "lse": lse, "cache": s["cache"]}
    if path == "indexer":
        ops.index_key_store(s["new"], s["slots"], s["keys"])
        scores = ops.indexer_scores(s["q"], s["w"], s["keys"], s["table"], s["limits"], s["width"])
        return {"scores": scores, "positions": ops.topk_positions(scores, min(c["K"], s["width"])), "keys": s["keys"]}
    if path == "prefill":
        ops.kv_store_mha(s["kn"], s["vn"], s["slots"], s["kc"], s["vc"], s["ks"], s["vs"])
        out = ops.prefill_attention(s["q"], s["kc"], s["vc"], s["table"], s["start_d"], s["priors_d"],
                                    max_q_len=s["longest"], sm_scale=c["d"] ** -0.5, k_scale=s["ks"],
                                    v_scale=s["vs"], sinks=s["sinks"], window=c["window"])
        return {"out": out, "k": _raw(s["kc"]), "v": _raw(s["vc"])}
    q = ops.qkv_norm_rope_store(s["qkv"], cos=s["cos"], sin=s["sin"], num_q_heads=c["H"], num_kv_heads=c["G"],
                                d_head=c["d"], k_cache=s["kc"], v_cache=s["vc"], slot_mapping=s["slots"],
                                q_norm=s["gamma"][0], k_norm=s["gamma"][1], k_scale=s["ks"], v_scale=s["vs"])
    return {"out": q, "k": _raw(s["kc"]), "v": _raw(s["vc"])}


# ---- what a pass cannot do without ----

def work(case):
    c = case
    path = c["path"]
    esz = 1 if c.get("fp8") else 2
    if path in ("gqa", "gqa_multi"):
        S = c.get("S", 1)
        lens = [max(n, S) for n in _spread(c["lo"], c["hi"], c["B"])]
        prior = [n - S if not c["window"] else min(n - S, c["window"] - 1) for n in lens]
        seen = sum(S * (n - S) + S * (S + 1) // 2 if not c["window"] else sum(min(n - S + j + 1, c["window"])
                                                                              for j in range(S)) for n in lens)
        b = sum(prior) * c["G"] * c["d"] * 2 * esz + sum(-(-n // c["P"]) for n in prior) * 4
        b += c["B"] * S * (c["G"] * c["d"] * 2 * (2 + esz) + c["H"] * c["d"] * 4)
        return {"bytes": b, "flops": 4 * c["d"] * c["H"] * seen}
    if path == "mla":
        lens = _spread(c["lo"], c["hi"], c["B"])
        row = 580 if c["fp8"] else 1152
        b = (sum(lens) - c["B"]) * row + sum(-(-n // c["P"]) for n in lens) * 4
        b += c["B"] * (1152 + row + c["H"] * (576 + 512) * 2)
        return {"bytes": b, "flops": 2 * (576 + 512) * c["H"] * sum(lens)}
    if path == "dsa":
        spec = c["spec"]
        kept = [min(c["K"], n - spec) * spec for n in _spread(c["lo"], c["hi"], c["B"])]
        T = c["B"] * spec
        b = sum(kept) * (640 + 8) + T * (1152 + 640 + c["H"] * ((576 + 512) * 2 + 4))
        return {"bytes": b, "flops": 2 * (576 + 512) * c["H"] * (sum(kept) + T)}
    if path == "indexer":
        n = sum(_spread(c["lo"], c["hi"], c["B"]))
        b = n * 130 + c["B"] * (c["H"] * 260 + c["K"] * 4 + 384)
        return {"bytes": b, "flops": 2 * 128 * c["H"] * n}
    if path == "prefill":
        chunks, priors = _spread(c["lo"], c["hi"], c["R"]), _spread(c["prior_lo"], c["prior_hi"], c["R"])
        # which chunk meets which prior is the seed's: the mean over the pairings
        mean = sum(priors) / len(priors)
        if c["window"]:
            seen = sum(n * min(c["window"], mean + (n + 1) / 2) for n in chunks)
            prior = sum(min(c["window"], p) for p in priors)
        else:
            seen = sum(n * mean + n * (n + 1) / 2 for n in chunks)
            prior = sum(priors)
        T = sum(chunks)
        b = prior * c["G"] * c["d"] * 2 * esz + T * (c["G"] * c["d"] * 2 * (2 + esz) + c["H"] * c["d"] * 4)
        return {"bytes": b, "flops": 4 * c["d"] * c["H"] * seen}
    d, width = c["d"], (c["H"] + 2 * c["G"]) * c["d"]
    return {"bytes": c["T"] * (width * 2 + 4 * d + 8 + c["H"] * d * 2 + 2 * c["G"] * d * esz), "flops": 0}


def tolerance(case):
    """Outputs in bf16 with fp32 accumulation over bf16 probabilities; pool bytes and positions are whole numbers and
    stay the same. About four times what each path shows against 64 bits."""
    return {"rel": {"gqa": 9e-3, "gqa_multi": 9e-3, "mla": 8e-3, "dsa": 8e-3, "indexer": 6.4e-3, "prefill": 9e-3,
                    "qkv": 1.3e-2}[case["path"]], "max": 0.1}


# ---- the same in 64 bits ----

def _dequant(t, s, multiply):
    t = t.double()
    if s is None:
        return t
    s = s.double().reshape(1, -1, *([1] * (t.dim() - 2)))
    return t / s if multiply else t * s


def _as_stored(x, s, multiply):
    """[n, G, d] new tokens as the pool holds them, in 64 bits."""
    if s is None:
        return x.double()
    r = s.reshape(1, -1, 1)
    if multiply:
        return (x * r.to(torch.bfloat16)).clamp(-448, 448).to(FP8).double() / r.double()
    return (x.float() / r).clamp(-448, 448).to(FP8).double() * r.double()


def _attend(q, k, v, seen, scale, sinks):
    """q [S, H, d], k / v [n, G, d] in 64 bits, seen [S, n]: softmax attention [S, H, d]."""
    S, H, d = q.shape
    G = k.shape[1]
    out = torch.empty(S, H, d, dtype=torch.float64, device=DEV)
    for g in range(G):
        heads = slice(g * (H // G), (g + 1) * (H // G))
        scores = (q[:, heads].reshape(-1, d) @ k[:, g].T.contiguous()).reshape(S, H // G, -1) * scale
        scores = scores.masked_fill(~seen[:, None], -math.inf)
        if sinks is not None:
            col = sinks[heads].double()[None, :, None].expand(S, -1, 1)
            p = torch.softmax(torch.cat([scores, col], dim=-1), dim=-1)[..., :-1]
        else:
            p = torch.softmax(scores, dim=-1)
        out[:, heads] = (p.reshape(-1, p.shape[-1]) @ v[:, g].contiguous()).reshape(S, H // G, d)
    return out


def _gather(cache, table_row, n, P):
    """[n, G, d] of a request's first n positions."""
    pages = table_row[:-(-n // P)].long() if n else table_row[:0].long()
    return cache[pages].transpose(1, 2).reshape(-1, cache.shape[1], cache.shape[3])[:n]


def exact(case, seed):
    c = case
    s = _inputs(case, seed)
    path = c["path"]
    if path in ("gqa", "gqa_multi", "prefill"):
        multiply = bool(c["fp8"] and c.get("sinks") and path != "prefill")
        out = []
        for r in range(len(s["table"])):
            if path == "prefill":
                a, b = s["start"][r], s["start"][r + 1]
                prior, q, kn, vn = s["priors"][r], s["q"][a:b], s["kn"][a:b], s["vn"][a:b]
            else:
                q, kn, vn = s["q"][r], s["kn"][r], s["vn"][r]
                prior = s["lens"][r] - q.shape[0]
            S = q.shape[0]
            k, v = (torch.cat([_dequant(_gather(cache, s["table"][r], prior, c["P"]), sc, multiply),
                               _as_stored(new, sc, multiply)])
                    for cache, sc, new in ((s["kc"], s["ks"], kn), (s["vc"], s["vs"], vn)))
            at, pos = torch.arange(prior + S, device=DEV), torch.arange(prior, prior + S, device=DEV)[:, None]
            seen = at <= pos
            if c["window"]:
                seen &= at > pos - c["window"]
            out.append(_attend(q.double(), k, v, seen, c["d"] ** -0.5, s["sinks"]))
        out = torch.cat(out) if path == "prefill" else torch.stack(out)
        return {"out": out[:, 0].contiguous() if path == "gqa" else out, "k": None, "v": None}
    if path == "mla":
        out = []
        for b, n in enumerate(s["lens"]):
            at = torch.arange(n - 1, device=DEV)
            rows = _slots(s["table"], torch.full_like(at, b), at, c["P"])
            if c["fp8"]:
                hist = s["cache"][rows].view(FP8).double() * s["sc"][rows].double()[:, None]
                x = s["new"][b].float()
                sc = x.abs().max() / 448
                own = (x / sc).clamp(-448, 448).to(FP8).double() * sc.double()
            else:
                hist, own = s["cache"][rows].double(), s["new"][b].double()
            keys = torch.cat([hist, own[None]])
            q = torch.cat([s["ql"][b], s["qp"][b]], dim=1).double()
            p = torch.softmax((q @ keys.T.contiguous()) * 192 ** -0.5, dim=-1)
            out.append(p @ keys[:, :512].contiguous())
        return {"out": torch.stack(out), "cache": None, "scale": None}
    if path == "dsa":
        # latent dim 256 a + 128 b + p lies at byte 128 + 256 a + 2 p + b of a 640-byte row
        dim = torch.arange(512, device=DEV)
        byte = 128 + 256 * (dim // 256) + 2 * (dim % 128) + (dim % 256) // 128
        scale, spec = s["scale"], c["spec"]

        def values(rows):
            return torch.cat([rows[:, byte].view(FP8).double() * scale,
                              rows[:, :128].contiguous().view(torch.bfloat16).double() * scale], dim=1)

        own = s["own"].float()
        own = torch.cat([(own[:, 64:] / scale).clamp(-448, 448).to(FP8).double() * scale,
                         (own[:, :64] / scale).to(torch.bfloat16).double() * scale], dim=1)
        out, lse = [], []
        for t in range(s["idx"].shape[0]):
            b = t // spec
            sel = s["idx"][t][s["idx"][t] >= 0].long()
            keys = [values(s["cache"][_slots(s["table"], torch.full_like(sel, b), sel, c["P"])]),
                    own[b * spec:t + 1]]
            keys = torch.cat(keys)
            q = torch.cat([s["qa"][t], s["qp"][t]], dim=1).double()
            scores = (q @ keys.T.contiguous()) * 0.0625
            out.append(torch.softmax(scores, dim=-1) @ keys[:, :512].contiguous())
            lse.append(torch.logsumexp(scores, dim=-1))
        return {"out": torch.stack(out), "lse": torch.stack(lse), "cache": None}
    if path == "indexer":
        scores = torch.full((c["B"], s["width"]), -1e30, dtype=torch.float64, device=DEV)
        for b, n in enumerate(s["limits"].tolist()):
            at = torch.arange(n, device=DEV)
            rows = _slots(s["table"], torch.full_like(at, b), at, c["P"])
            keys = s["keys"].reshape(-1, 128)[rows].view(FP8).double()
            raw = torch.relu(s["q"][b].double() @ keys.T.contiguous()) * 128 ** -0.5
            scores[b, :n] = (s["w"][b].double()[None] @ raw)[0]
        return {"scores": scores, "positions": None, "keys": None}
    T, H, G, d = c["T"], c["H"], c["G"], c["d"]
    q = s["qkv"][:, :H * d].double().reshape(T, H, d)
    if c["norm"]:
        q = q * torch.rsqrt((q * q).mean(-1, keepdim=True) + 1e-6) * s["gamma"][0].double()
    turned = torch.cat([-q[..., d // 2:], q[..., :d // 2]], dim=-1)
    return {"out": q * s["cos"].double()[:, None] + turned * s["sin"].double()[:, None], "k": None, "v": None}
