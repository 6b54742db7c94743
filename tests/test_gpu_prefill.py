"""Segmented prefill attention over the FP8 or bf16 pool (ops.prefill_attention, the reference's segmented_attention) against
the CPU oracle (oracle/attention.segmented_prefill) on the same pool bytes: within the attention bar."""

from __future__ import annotations

import random

import pytest
import torch

from conftest import announce
from _harness import assert_close_attn
from oracle import attention as oatt
from sglang_neuron_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(seed, H, G, d, P, priors, lens, spare_pages=5, bf16=False):
    """A pool holding every request's prior and chunk (stored by ops.kv_store_mha with per-head absmax scales), its
    table, the chunk queries and their row offsets."""
    g = torch.Generator().manual_seed(seed)
    R = len(priors)
    spans = [p + s for p, s in zip(priors, lens)]
    pages = [-(-x // P) for x in spans]
    nb = sum(pages) + spare_pages + 1
    width = max(pages) + 2
    perm = torch.randperm(nb - 1, generator=g) + 1
    table = torch.full((R, width), -1, dtype=torch.int32)
    used = 0
    for r, n in enumerate(pages):
        table[r, :n] = perm[used:used + n].to(torch.int32)
        used += n
    k_tok = [torch.randn(x, G, d, generator=g).to(torch.bfloat16) for x in spans]
    v_tok = [torch.randn(x, G, d, generator=g).to(torch.bfloat16) for x in spans]
    k_all, v_all = torch.cat(k_tok), torch.cat(v_tok)
    ks = (k_all.float().abs().amax(dim=(0, 2)) / 448.0).clamp(min=1e-6)
    vs = (v_all.float().abs().amax(dim=(0, 2)) / 448.0).clamp(min=1e-6)
    slots = torch.cat([table[r, torch.arange(x) // P].to(torch.int64) * P + torch.arange(x) % P
                       for r, x in enumerate(spans)])
    kc = torch.zeros(nb, G, P, d, dtype=torch.bfloat16 if bf16 else torch.float8_e4m3fn, device=DEV)
    vc = torch.zeros_like(kc)
    if bf16:
        ks = vs = None
        ops.kv_store_mha(k_all.to(DEV), v_all.to(DEV), slots.to(DEV), kc, vc)
    else:
        ops.kv_store_mha(k_all.to(DEV), v_all.to(DEV), slots.to(DEV), kc, vc, ks.to(DEV), vs.to(DEV))
    T = sum(lens)
    q = torch.randn(T, H, d, generator=g).to(torch.bfloat16)
    q_start = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    return q, kc, vc, ks, vs, table, q_start, torch.tensor(priors, dtype=torch.int32)


def _unsplit(q, kc, vc, ks, vs, table, q_start, priors, longest, scale, window=0, sinks=None):
    """sna_prefill_attention: the entry without a workspace, which never splits. Device tensors."""
    lib = _lib.load()
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    out = torch.empty_like(q)
    rc = lib.sna_prefill_attention(ptr(q), ptr(kc), ptr(vc), ptr(ks), ptr(vs), ptr(table), table.stride(0), table.shape[1],
                                   ptr(q_start), ptr(priors), priors.numel(), longest, ptr(sinks), scale, window, ptr(out),
                                   q.shape[1], kc.shape[1], q.shape[2], kc.shape[2], kc.shape[0],
                                   _lib.DTYPE_BF16 if ks is None else _lib.DTYPE_FP8_E4M3FN,
                                   torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    return out


CASES = [
    ("qwen3-8b-chunks", 1, dict(H=32, G=8, d=128, P=16, priors=(0, 100, 1000), lens=(64, 200, 37)), 0, False),
    ("gpt-oss-swa-sinks", 2, dict(H=8, G=1, d=64, P=16, priors=(300, 0), lens=(150, 129)), 128, True),
    ("group3-page64", 3, dict(H=12, G=4, d=64, P=64, priors=(70, 5), lens=(33, 90)), 0, True),
    ("long-prior", 4, dict(H=8, G=2, d=128, P=16, priors=(40000,), lens=(8,)), 0, False),
    ("window-1000-page32", 5, dict(H=16, G=4, d=128, P=32, priors=(5000,), lens=(300,)), 1000, False),
    ("mha-d128", 6, dict(H=4, G=4, d=128, P=16, priors=(17, 250), lens=(140, 3)), 0, False),
    ("empty-request", 7, dict(H=8, G=2, d=64, P=16, priors=(40, 9, 0), lens=(20, 0, 33)), 0, False),
    ("bf16-qwen3-0.6b", 8, dict(H=16, G=8, d=128, P=16, priors=(0, 300, 77), lens=(128, 45, 200), bf16=True), 0, False),
    ("bf16-swa-sinks-d64", 10, dict(H=8, G=2, d=64, P=32, priors=(500, 3), lens=(70, 130), bf16=True), 96, True),
    ("bf16-long-prior", 11, dict(H=4, G=1, d=128, P=16, priors=(34000,), lens=(20,), bf16=True), 0, False),
    ("fp8-long-window-page64", 13, dict(H=16, G=4, d=128, P=64, priors=(70000, 3000), lens=(100, 70)), 40000, True),
    # pages that are multiples of 16 but not powers of two (the tile's page lookups divide)
    ("fp8-page48-window", 14, dict(H=16, G=4, d=128, P=48, priors=(3000, 7), lens=(90, 60)), 500, False),
    ("bf16-page48-sinks", 15, dict(H=8, G=2, d=64, P=48, priors=(100,), lens=(70,), bf16=True), 0, True),
]


@pytest.mark.parametrize("name,seed,cfg,window,sinks", CASES, ids=[c[0] for c in CASES])
def test_prefill_attention_matches_oracle(name, seed, cfg, window, sinks):
    """Each case as the package calls it (long priors split their keys) and through the entry that never splits, whose
    workgroups then walk every key: more than the block-table entries staged at a time (2047 pages) in the long cases."""
    announce(f"prefill {name}: {cfg} window={window} sinks={sinks}")
    q, kc, vc, ks, vs, table, q_start, priors = _case(seed, **cfg)
    H, d = cfg["H"], cfg["d"]
    sk = torch.randn(H, generator=torch.Generator().manual_seed(seed + 50)) if sinks else None
    scale = d ** -0.5
    bf16 = cfg.get("bf16", False)
    longest = max(cfg["lens"]) + 7
    kd, vd = (None, None) if bf16 else (ks.to(DEV), vs.to(DEV))
    skd = None if sk is None else sk.to(DEV)
    args = (q.to(DEV), kc, vc, table.to(DEV), q_start.to(DEV), priors.to(DEV))
    out = ops.prefill_attention(*args, max_q_len=longest, sm_scale=scale, k_scale=kd, v_scale=vd, sinks=skd, window=window)
    whole = _unsplit(*args[:3], kd, vd, *args[3:], longest, scale, window, skd)
    torch.cuda.synchronize()
    kh, vh = (kc.cpu(), vc.cpu()) if bf16 else (kc.cpu().view(torch.uint8), vc.cpu().view(torch.uint8))
    want = oatt.segmented_prefill(q, kh, vh, table, q_start, priors, sm_scale=scale, k_scale=ks, v_scale=vs, sinks=sk,
                                  window=window)
    assert_close_attn(out.cpu(), want, name)
    assert_close_attn(whole.cpu(), want, f"{name} unsplit")


def _random_shape(seed: int):
    r = random.Random(seed)
    G = r.choice([1, 2, 4, 8])
    group = r.choice([g for g in (1, 2, 4, 8, 16) if G * g <= 64])
    R = r.randint(1, 3)
    cfg = dict(H=G * group, G=G, d=r.choice([64, 128]), P=r.choice([16, 32, 48, 64, 128]),
               priors=tuple(r.randint(0, 3000) for _ in range(R)), lens=tuple(r.randint(1, 200) for _ in range(R)),
               bf16=r.random() < 0.35)
    return cfg, r.choice([0, 0, r.randint(16, 1500)]), r.random() < 0.4


RANDOM_SEEDS = list(range(9400, 9410))


@pytest.mark.parametrize("seed", RANDOM_SEEDS)
def test_prefill_random_shape(seed):
    """Seeded random shapes (groups, head dims, pages including non-powers of two, requests, windows, sinks, FP8 and
    bf16 pools), drawn once from fixed seeds, against the oracle."""
    cfg, window, sinks = _random_shape(seed)
    test_prefill_attention_matches_oracle(f"random-{seed}", seed, cfg, window, sinks)


# the split's edges: one tile past the least table that splits, a block's keys cut into many splits, splits under a window, a
# group that does not divide a block's rows, chunks of unequal length (query blocks that do not exist), as many blocks as a
# split launch takes, a wide table over keys too few to pay (the device drops the split)
SPLIT_CASES = [
    ("seventeen-tiles", 21, dict(H=8, G=2, d=128, P=16, priors=(1025, 0), lens=(60, 5)), 0, False, 3),
    ("forty-tiles", 27, dict(H=8, G=2, d=128, P=16, priors=(2500, 1030), lens=(60, 5)), 0, False, 5),
    ("many-splits-d64", 22, dict(H=4, G=1, d=64, P=16, priors=(20000, 3), lens=(9, 70)), 0, True, 40),
    ("window-splits-bf16", 23, dict(H=8, G=1, d=128, P=64, priors=(9000, 700), lens=(40, 30), bf16=True), 3000, True, 6),
    ("group3-splits", 24, dict(H=6, G=2, d=64, P=48, priors=(2500,), lens=(43,), bf16=True), 0, False, 5),
    ("most-blocks", 25, dict(H=16, G=8, d=64, P=16, priors=(1600, 0), lens=(33, 1024)), 0, False, 4),
    ("dropped", 28, dict(H=8, G=2, d=128, P=16, priors=(600, 30), lens=(60, 5)), 0, True, 1),
]


def _splits_run(ws, slots, R, blocks, G, d):
    """The split count of every (KV head, request, query block) a split launch left in its workspace (blocks a request does
    not have keep what the workspace held)."""
    at = slots * 128 * (d + 2) * 4
    return ws[at:at + 8 * G * R * blocks].view(torch.int32).reshape(G, R, blocks, 2)[..., 1].cpu()


@pytest.mark.parametrize("name,seed,cfg,window,sinks,most", SPLIT_CASES, ids=[c[0] for c in SPLIT_CASES])
def test_prefill_split_edges(name, seed, cfg, window, sinks, most):
    """Launches that may split the keys, at the sizes where a split can go wrong; then the same call through the entry that
    takes no workspace (which never splits): both within the attention bar of the oracle. most: at least so many splits of
    a query block ran, or (1) the device dropped the split."""
    announce(f"prefill split {name}: {cfg} window={window} sinks={sinks}")
    q, kc, vc, ks, vs, table, q_start, priors = _case(seed, **cfg)
    if most == 1:
        table = torch.cat([table, torch.full((len(table), 200), -1, dtype=torch.int32)], dim=1)
    H, G, d, P, bf16 = cfg["H"], cfg["G"], cfg["d"], cfg["P"], cfg.get("bf16", False)
    R, longest, width = len(cfg["lens"]), max(cfg["lens"]), table.shape[1]
    sk = torch.randn(H, generator=torch.Generator().manual_seed(seed + 50)) if sinks else None
    lib = _lib.load()
    assert lib.sna_prefill_workspace_bytes(R, longest, H, G, d, P, width, window) > 0
    qd, td, sd, pd = q.to(DEV), table.to(DEV), q_start.to(DEV), priors.to(DEV)
    ksd, vsd = (None, None) if bf16 else (ks.to(DEV), vs.to(DEV))
    skd = None if sk is None else sk.to(DEV)
    kh, vh = (kc.cpu(), vc.cpu()) if bf16 else (kc.cpu().view(torch.uint8), vc.cpu().view(torch.uint8))
    want = oatt.segmented_prefill(q, kh, vh, table, q_start, priors, sm_scale=d ** -0.5, k_scale=ks, v_scale=vs,
                                  sinks=sk, window=window)
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    need = lib.sna_prefill_workspace_bytes(R, longest, H, G, d, P, width, window)
    blocks = -(-longest // (128 // (H // G)))
    slots = (need - 8 * G * R * blocks) // (128 * (d + 2) * 4)
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
    out = torch.empty_like(qd)
    rc = lib.sna_prefill_attention_split(
        ptr(qd), ptr(kc), ptr(vc), ptr(ksd), ptr(vsd), ptr(td), td.stride(0), width, ptr(sd), ptr(pd), R, longest, ptr(skd),
        d ** -0.5, window, ptr(out), H, G, d, P, kc.shape[0], _lib.DTYPE_BF16 if bf16 else _lib.DTYPE_FP8_E4M3FN, ptr(ws),
        need, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    assert_close_attn(out.cpu(), want, name)
    counts = _splits_run(ws, slots, R, blocks, G, d)
    for r, n in enumerate(cfg["lens"]):  # a request's query blocks have splits, no others do
        assert bool(((counts[:, r] > 0) == (torch.arange(blocks) < -(-n // (128 // (H // G))))).all()), counts
    assert int(counts.max()) >= most if most > 1 else int(counts.max()) == 1, counts
    packed = ops.prefill_attention(qd, kc, vc, td, sd, pd, max_q_len=longest, sm_scale=d ** -0.5, k_scale=ksd, v_scale=vsd,
                                   sinks=skd, window=window)
    assert torch.equal(packed, out)
    whole = _unsplit(qd, kc, vc, ksd, vsd, td, sd, pd, longest, d ** -0.5, window, skd)
    torch.cuda.synchronize()
    assert_close_attn(whole.cpu(), want, f"{name} unsplit")


@pytest.mark.parametrize("bf16", [False, True], ids=["fp8", "bf16"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("P", [16, 48, 64])
def test_prefill_one_tile(P, d, bf16):
    """Prompts whose tables name at most 64 keys (a kernel of their own): within the attention bar of the oracle, and the
    bits of the general kernel over a wider table, with NaN in every slot no query may see and pages of -1 past the prompt."""
    announce(f"prefill one tile P={P} d={d} bf16={bf16}")
    H, G = 8, 2
    for lens, window in (((1,), 0), ((16, 3), 0), ((17, 32), 5), ((33,), 0), ((48, 1, 20), 0), ((49, 63), 40), ((64,), 0)):
        if max(lens) > 64 // P * P:
            continue
        n, R = max(lens), len(lens)
        q, kc, vc, ks, vs, table, q_start, priors = _case(51 + n, H=H, G=G, d=d, P=P, priors=(0,) * R, lens=lens, bf16=bf16)
        used = torch.zeros(kc.shape[0] * P, dtype=torch.bool)
        for r, m in enumerate(lens):
            at = torch.arange(m)
            used[table[r, at // P].long() * P + at % P] = True
        dead = (~used).reshape(kc.shape[0], 1, P, 1).to(DEV)
        kh, vh = (kc.cpu(), vc.cpu()) if bf16 else (kc.cpu().view(torch.uint8), vc.cpu().view(torch.uint8))
        for cache in (kc, vc):
            cache.view(torch.int16 if bf16 else torch.uint8).masked_fill_(dead, 0x7FC0 if bf16 else 0x7F)
        want = oatt.segmented_prefill(q, kh, vh, table, q_start, priors, sm_scale=d ** -0.5, k_scale=ks, v_scale=vs,
                                      sinks=None, window=window)
        kd, vd = (None, None) if bf16 else (ks.to(DEV), vs.to(DEV))
        qd, sd, pd = q.to(DEV), q_start.to(DEV), priors.to(DEV)
        narrow = table[:, :-(-n // P)].contiguous().to(DEV)
        assert narrow.shape[1] * P <= 64
        out = ops.prefill_attention(qd, kc, vc, narrow, sd, pd, max_q_len=n, sm_scale=d ** -0.5, k_scale=kd, v_scale=vd,
                                    window=window)
        assert_close_attn(out.cpu(), want, f"{lens}")
        wide = torch.full((R, 8), -1, dtype=torch.int32)
        wide[:, :min(8, table.shape[1])] = table[:, :8]
        assert torch.equal(out, _unsplit(qd, kc, vc, kd, vd, wide.to(DEV), sd, pd, n, d ** -0.5, window)), lens


@pytest.mark.parametrize("bf16", [False, True], ids=["fp8", "bf16"])
@pytest.mark.parametrize("prior", [70, 2500], ids=["whole", "split"])
def test_prefill_ignores_unused_slots_and_invalid_pages(bf16, prior):
    """NaN in every slot no query may see (page 0, the last page's tail, unused pages, a page the table marks invalid)
    does not reach the output: against a float64 attention over the visible keys."""
    announce(f"prefill nan slots bf16={bf16} prior={prior}")
    H, G, d, P, n = 8, 2, 64, 16, 21
    q, kc, vc, ks, vs, table, q_start, priors = _case(31, H=H, G=G, d=d, P=P, priors=(prior,), lens=(n,), bf16=bf16)
    span = prior + n
    hole = 3  # the page of keys 48 .. 63
    table[0, hole] = -1
    pos = torch.arange(span)
    live = pos // P != hole
    slots = (table[0, pos // P].to(torch.int64) * P + pos % P)[live]
    used = torch.zeros(kc.shape[0] * P, dtype=torch.bool)
    used[slots] = True
    dead = (~used).reshape(kc.shape[0], 1, P, 1).to(DEV)
    raw = torch.int16 if bf16 else torch.uint8
    for cache in (kc, vc):
        cache.view(raw).masked_fill_(dead, 0x7FC0 if bf16 else 0x7F)
    one = (torch.ones(G), torch.ones(G)) if bf16 else (ks, vs)
    k, v = ((c.cpu().float().permute(0, 2, 1, 3).reshape(-1, G, d)[slots] * s.reshape(1, G, 1)).double()
            for c, s in zip((kc, vc), one))
    qh = q.double().reshape(n, G, H // G, d)
    scores = torch.stack([torch.einsum("sjd,kd->sjk", qh[:, g], k[:, g]) for g in range(G)], 1) * d ** -0.5
    seen = pos[live][None, :] <= (prior + torch.arange(n))[:, None]
    p = torch.softmax(scores.masked_fill(~seen[:, None, None], float("-inf")), -1)
    want = torch.stack([torch.einsum("sjk,kd->sjd", p[:, g], v[:, g]) for g in range(G)], 1).reshape(n, H, d)
    out = ops.prefill_attention(q.to(DEV), kc, vc, table.to(DEV), q_start.to(DEV), priors.to(DEV), max_q_len=n,
                                sm_scale=d ** -0.5, k_scale=None if bf16 else ks.to(DEV),
                                v_scale=None if bf16 else vs.to(DEV))
    torch.cuda.synchronize()
    assert_close_attn(out.cpu(), want, "nan slots")


def test_prefill_split_ignores_lengths_it_cannot_hold():
    """In a launch that splits, a padding request (no token) and one whose prior is below zero (no visible key: its rows
    are what the unsplit entry writes) leave the other requests' splits and outputs as they are without them."""
    announce("prefill split padding requests")
    H, G, d, P = 8, 2, 64, 16
    q, kc, vc, ks, vs, table, _, _ = _case(41, H=H, G=G, d=d, P=P, priors=(2500, 0, 0), lens=(40, 0, 16))
    dev = [t.to(DEV) for t in (ks, vs)]
    q_start = torch.tensor([0, 40, 40, 56], dtype=torch.int32, device=DEV)
    lib = _lib.load()

    def run(n, priors):
        R = len(priors)
        assert lib.sna_prefill_workspace_bytes(R, 40, H, G, d, P, table.shape[1], 0) > 0
        return ops.prefill_attention(q[:n].to(DEV), kc, vc, table[:R].to(DEV), q_start[:R + 1],
                                     torch.tensor(priors, dtype=torch.int32, device=DEV), max_q_len=40, sm_scale=0.125,
                                     k_scale=dev[0], v_scale=dev[1]).cpu()

    alone = run(40, [2500])
    for low in (-300, -64, -5000):
        both = run(56, [2500, low, low])
        assert torch.equal(both[:40], alone), low
        assert bool(torch.isnan(both[40:].float()).all()), low  # softmax over no key


@pytest.mark.parametrize("bf16", [False, True], ids=["fp8", "bf16"])
@pytest.mark.parametrize("prior", [0, 1500], ids=["whole", "split"])
def test_prefill_widest_window_is_no_window(bf16, prior):
    """A window of up to 2^31 - 1 keys holds every key of any row: the outputs are those of no window."""
    announce(f"prefill widest window bf16={bf16} prior={prior}")
    H, G, d, P, n = 8, 2, 64, 16, 70
    q, kc, vc, ks, vs, table, q_start, priors = _case(43, H=H, G=G, d=d, P=P, priors=(prior,), lens=(n,), bf16=bf16)
    kw = dict(max_q_len=n, sm_scale=0.125, k_scale=None if bf16 else ks.to(DEV), v_scale=None if bf16 else vs.to(DEV))
    args = (q.to(DEV), kc, vc, table.to(DEV), q_start.to(DEV), priors.to(DEV))
    none = ops.prefill_attention(*args, **kw)
    for window in (2**31 - 1, 2**31 - 4, 2**31 - 64, 1 << 20):
        assert torch.equal(ops.prefill_attention(*args, window=window, **kw), none), window


def test_prefill_split_workspace_refusals():
    """A workspace smaller than the split needs, or not 16-byte aligned, is refused before any launch."""
    q, kc, vc, ks, vs, table, q_start, priors = _case(26, H=8, G=2, d=64, P=16, priors=(1900,), lens=(20,))
    lib = _lib.load()
    need = lib.sna_prefill_workspace_bytes(1, 20, 8, 2, 64, 16, table.shape[1], 0)
    ws = torch.empty(need + 16, dtype=torch.uint8, device=DEV)
    d = [t.to(DEV) for t in (q, ks, vs, table, q_start, priors)]
    out = torch.empty_like(d[0])

    def call(ptr, n):
        return lib.sna_prefill_attention_split(
            d[0].data_ptr(), kc.data_ptr(), vc.data_ptr(), d[1].data_ptr(), d[2].data_ptr(), d[3].data_ptr(),
            d[3].stride(0), table.shape[1], d[4].data_ptr(), d[5].data_ptr(), 1, 20, None, 0.125, 0, out.data_ptr(), 8, 2,
            64, 16, kc.shape[0], _lib.DTYPE_FP8_E4M3FN, ptr, n, torch.cuda.current_stream().cuda_stream)

    assert need > 0 and call(ws.data_ptr(), need) == 0
    assert call(ws.data_ptr(), need - 1) == _lib.SNA_ERR_WORKSPACE
    assert call(ws.data_ptr() + 4, need) == _lib.SNA_ERR_INVALID_ARGUMENT
    torch.cuda.synchronize()


def test_segmented_attention_reference_signature():
    """ops.segmented_attention takes the reference's arguments (one request, q [heads, S, d], sink [heads, 1])."""
    announce("prefill segmented_attention signature")
    q, kc, vc, ks, vs, table, q_start, priors = _case(9, H=8, G=2, d=128, P=16, priors=(77,), lens=(50,))
    sk = torch.randn(8, 1)
    out = ops.segmented_attention(q.transpose(0, 1).contiguous().to(DEV), k_cache=kc, v_cache=vc,
                                  block_tables=table.to(DEV), prior_tokens=torch.tensor([[77]]), block_size=16,
                                  kv_segment_size=512, scale=0.1, sliding_window=None, sink=sk.to(DEV),
                                  k_scale=ks.to(DEV), v_scale=vs.to(DEV))
    torch.cuda.synchronize()
    assert out.shape == (8, 50, 128)
    want = oatt.segmented_prefill(q, kc.cpu().view(torch.uint8), vc.cpu().view(torch.uint8), table, q_start, priors,
                                  sm_scale=0.1, k_scale=ks, v_scale=vs, sinks=sk.reshape(-1))
    assert_close_attn(out.transpose(0, 1).cpu(), want, "segmented_attention")


def test_prefill_rejects_bad_pages_and_missing_scales():
    q = torch.zeros(4, 8, 64, dtype=torch.bfloat16, device=DEV)
    kc = torch.zeros(3, 2, 16, 64, dtype=torch.float8_e4m3fn, device=DEV)
    args = (q, kc, kc, torch.zeros(1, 2, dtype=torch.int32, device=DEV), torch.tensor([0, 4], dtype=torch.int32,
                                                                                      device=DEV),
            torch.tensor([0], dtype=torch.int32, device=DEV))
    one = torch.ones(2, device=DEV)
    with pytest.raises(ValueError):
        ops.prefill_attention(*args, max_q_len=4, sm_scale=1.0)  # an FP8 pool without its scales
    kc8 = torch.zeros(3, 2, 8, 64, dtype=torch.float8_e4m3fn, device=DEV)
    with pytest.raises(ValueError):
        ops.prefill_attention(q, kc8, kc8, *args[3:], max_q_len=4, sm_scale=1.0, k_scale=one, v_scale=one)
    # more workgroups than the kernel numbers in 32 bits: refused before any launch
    many = 65535
    with pytest.raises(ValueError, match="exceed the grid"):
        ops.prefill_attention(q, kc, kc, torch.zeros(many, 2, dtype=torch.int32, device=DEV),
                              torch.zeros(many + 1, dtype=torch.int32, device=DEV),
                              torch.zeros(many, dtype=torch.int32, device=DEV), max_q_len=2 ** 31 - 1, sm_scale=1.0,
                              k_scale=one, v_scale=one)


def test_prefill_takes_int64_tables_and_checks_host_offsets():
    """An int64 block table, q_start and prior_lens are converted (as the decode wrappers do); with a host copy of
    q_start, offsets that do not run from 0 to T or a chunk past max_q_len are refused before the launch."""
    announce("prefill int64 operands and host offsets")
    q, kc, vc, ks, vs, table, q_start, priors = _case(12, H=8, G=2, d=64, P=16, priors=(30, 5), lens=(40, 25))
    args = dict(max_q_len=40, sm_scale=0.125, k_scale=ks.to(DEV), v_scale=vs.to(DEV))
    out = ops.prefill_attention(q.to(DEV), kc, vc, table.to(torch.int64).to(DEV), q_start.to(torch.int64).to(DEV),
                                priors.to(torch.int64).to(DEV), host_q_start=q_start, **args)
    torch.cuda.synchronize()
    want = oatt.segmented_prefill(q, kc.cpu().view(torch.uint8), vc.cpu().view(torch.uint8), table, q_start, priors,
                                  sm_scale=0.125, k_scale=ks, v_scale=vs)
    assert_close_attn(out.cpu(), want, "int64 operands")
    dev_args = (q.to(DEV), kc, vc, table.to(DEV), q_start.to(DEV), priors.to(DEV))
    with pytest.raises(ValueError, match="max_q_len"):
        ops.prefill_attention(*dev_args, host_q_start=q_start, **{**args, "max_q_len": 39})
    with pytest.raises(ValueError, match="from 0 to T"):
        ops.prefill_attention(*dev_args, host_q_start=q_start - 1, **args)
