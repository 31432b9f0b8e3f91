"""Workloads of the paged int8 attention and of its cache writer, each as one
pass through the public entry points: the torch op, the slice builder with its
forward (what a serving engine calls once per layer) and the cache writer.

``listed()`` names the workloads, ``draw(rng)`` gives another one of the same
ranges, ``prepare`` makes a workload's inputs on the GPU, ``run`` makes one
pass, ``exact`` gives the same outputs in 64 bits from plain torch, ``work``
the bytes and operations of a pass, and ``tolerance`` how far two correct
implementations may lie apart.

An attention workload is a batch of decode-like requests (``decodes`` of
``q`` query tokens, context ``len_lo``..``len_hi``) and of prefill chunks
(``chunks`` of ``chunk_lo``..``chunk_hi`` query tokens behind a prefix of
``prefix_lo``..``prefix_hi`` cached tokens); the lengths are drawn from
``len_seed``, so that a workload's work is a property of the workload.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "pth-flash-attn_amd" / "python"))

from pth_flash_attn import ops, planner  # noqa: E402
from pth_flash_attn.cache import build_cache, carve_views, cell_bytes, make_queries  # noqa: E402
from pth_flash_attn.slices import SliceBuilder, run_slices  # noqa: E402

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
MAX_NUM_SEQS = 64  # the engine's batch bound that its workspace is reserved for


def _attn(name=None, **kw):
    """An attention workload: 32 q / 8 KV heads, D = 128, bf16, causal, pages
    of 16 slots, unless said otherwise."""
    case = {"kind": "attention", "Hq": 32, "Hkv": 8, "D": 128, "block": 16, "layout": "NHD",
            "dtype": "bf16", "window": 0, "causal": True, "one_launch": False,
            "decodes": 0, "q": 1, "len_lo": 1, "len_hi": 1,
            "chunks": 0, "chunk_lo": 1, "chunk_hi": 1, "prefix_lo": 0, "prefix_hi": 0,
            "len_seed": 1}
    case.update(kw)
    return case if name is None else {"name": name, **case}


def _write(name=None, **kw):
    """A cache write: keys and values of ``tokens`` tokens, cut from the fused
    projection's output, into their cells."""
    case = {"kind": "write", "tokens": 1, "Hq": 32, "Hkv": 8, "D": 128, "block": 16,
            "layout": "NHD", "dtype": "bf16"}
    case.update(kw)
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # One short chat request, one tensor-parallel shard: latency alone.
        _attn("decode_1x1k", Hq=4, Hkv=1, decodes=1, len_lo=1024, len_hi=1024),
        # A full decode batch of a served model: the headline workload.
        _attn("decode_64x32k", decodes=64, len_lo=1024, len_hi=32768, len_seed=2024),
        # One very long request, speculative verify of 4 drafted tokens.
        _attn("verify4_1x128k", decodes=1, q=4, len_lo=131072, len_hi=131072),
        # Sliding-window layer, verify of 16 drafted tokens in 8 requests.
        _attn("window_verify16_8x64k", decodes=8, q=16, len_lo=8192, len_hi=65536, window=2048,
              len_seed=4044),
        # A drafter's windowed non-causal layer, one request, large pages.
        _attn("drafter_1x2k", Hq=16, Hkv=4, block=864, window=2048, causal=False, decodes=1, q=8,
              len_lo=2056, len_hi=2056),
        # Chunked prefill and decode mixed in one launch: the largest.
        _attn("mixed_4x2k_60", one_launch=True, decodes=60, len_lo=2048, len_hi=65536, chunks=4,
              chunk_lo=2048, chunk_hi=2048, prefix_hi=30 * 1024, len_seed=5055),
        # A serving step on half of a model's heads, as the engine's forward
        # makes it: a decode slice, then the slice of one prefill chunk.
        _attn("step_tp2_24_1x2k", Hq=16, Hkv=4, dtype="fp16", block=32, decodes=24, len_lo=500,
              len_hi=20000, chunks=1, chunk_lo=2011, chunk_hi=2011, prefix_lo=6101,
              prefix_hi=6101, len_seed=7),
        # Head size 256 with 6 query heads per KV head: long verify, and one
        # chunk of a prompt in pages of 816 slots.
        _attn("d256_verify4_1x128k", Hq=12, Hkv=2, D=256, decodes=1, q=4, len_lo=131072,
              len_hi=131072),
        _attn("d256_prefill_1x2k", Hq=12, Hkv=2, D=256, block=816, chunks=1, chunk_lo=2048,
              chunk_hi=2048, prefix_lo=4099, prefix_hi=4099),
        # Head size 64: a decode batch, and two chunks of a prompt.
        _attn("d64_decode_48x16k", D=64, dtype="fp16", decodes=48, len_lo=300, len_hi=16384,
              len_seed=48),
        _attn("d64_prefill_2x1k", D=64, chunks=2, chunk_lo=700, chunk_hi=1500, prefix_lo=0,
              prefix_hi=8000, len_seed=64),
        # The cache write of a prefill step's tokens.
        _write("write_8k", tokens=8192),
    ]


# (Hq, Hkv) by head size: whole models and their tensor-parallel shards.
HEADS = {
    64: [(16, 4), (32, 8), (64, 8)],
    128: [(4, 1), (8, 1), (16, 2), (16, 4), (32, 4), (32, 8), (64, 8)],
    256: [(6, 1), (12, 2), (16, 4), (16, 8), (24, 4)],
}
MOST_BYTES = 2.0e9
MOST_FLOPS = 1.2e12


def _log(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    D = rng.choice([64, 128, 128, 256])
    Hq, Hkv = rng.choice(HEADS[D])
    base = {"Hq": Hq, "Hkv": Hkv, "D": D, "dtype": rng.choice(["bf16", "bf16", "fp16"]),
            "layout": rng.choice(["NHD", "NHD", "NHD", "HND"]),
            "block": rng.choice([16, 16, 32, 64, 528, 816])}
    what = rng.choice(["decode", "verify", "prefill", "step", "window", "drafter", "write"])
    if what == "write":
        return _write(tokens=_log(rng, 1, 16384), **base)
    if what in ("window", "drafter") and D != 128:
        what = "verify"
    base["len_seed"] = rng.randrange(1, 1 << 30)
    while True:
        kw = dict(base)
        if what in ("decode", "verify", "step", "window"):
            kw["decodes"] = _log(rng, 1, MAX_NUM_SEQS)
            kw["len_hi"] = _log(rng, 64, 131072)
            kw["len_lo"] = _log(rng, 16, kw["len_hi"])
        if what in ("verify", "window"):
            kw["q"] = rng.randint(2, 16) if what == "window" else rng.randint(2, 8)
        if what == "window":
            kw["window"] = rng.choice([512, 1024, 2048, 4096])
        if what == "drafter":
            kw.update(window=rng.choice([1024, 2048, 4096]), causal=False, q=rng.randint(2, 16),
                      decodes=_log(rng, 1, 8), len_lo=64, len_hi=_log(rng, 2048, 65536))
        if what in ("prefill", "step"):
            kw["chunks"] = rng.randint(1, 4)
            kw["chunk_hi"] = _log(rng, 100, 4096)
            kw["chunk_lo"] = max(65, kw["chunk_hi"] // 2)
            kw["chunk_hi"] = max(kw["chunk_lo"], kw["chunk_hi"])
            kw["prefix_hi"] = rng.choice([0, _log(rng, 100, 30000)])
        case = _attn(**kw)
        w = work(case)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS:
            return case


def lengths(case):
    """(query tokens, context tokens) per request: the decode-like requests
    first, as an engine orders them; one launch of a mixed batch takes them in
    any order, and has them last."""
    rng = np.random.default_rng(case["len_seed"])
    dec = [int(x) for x in rng.integers(case["len_lo"], case["len_hi"] + 1, case["decodes"])]
    dec = [(case["q"], max(x, case["q"])) for x in dec]
    pre = []
    for _ in range(case["chunks"]):
        n = int(rng.integers(case["chunk_lo"], case["chunk_hi"] + 1))
        pre.append((n, n + int(rng.integers(case["prefix_lo"], case["prefix_hi"] + 1))))
    both = pre + dec if case["one_launch"] else dec + pre
    return [a for a, _ in both], [b for _, b in both]


def _visible(case, q, L):
    """First and one past the last key that each of a request's queries sees."""
    p = np.arange(L - q, L, dtype=np.int64)
    W = case["window"]
    lo = np.maximum(0, p - W + 1) if W else np.zeros(q, np.int64)
    hi = p if case["causal"] else np.minimum(L - 1, p + W - 1) if W else np.full(q, L - 1)
    return lo, hi + 1


def work(case):
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    if case["kind"] == "write":
        n = case["tokens"] * Hkv
        return {"bytes": n * (2 * D * 2 + cell_bytes(D)) + 8 * case["tokens"], "flops": 0}
    keys = pairs = tokens = pages = 0
    for q, L in zip(*lengths(case)):
        lo, hi = _visible(case, q, L)
        keys += int(hi[-1] - lo[0])
        pairs += int((hi - lo).sum())
        tokens += q
        pages += -(-int(hi[-1]) // case["block"]) - int(lo[0]) // case["block"]
    return {"bytes": keys * Hkv * cell_bytes(D) + 2 * tokens * Hq * D * 2 + 4 * pages,
            "flops": 4 * D * Hq * pairs}


def prepare(case, seed):
    if case["kind"] == "write":
        return _prepare_write(case, seed)
    q_lens, seq_lens = lengths(case)
    Hq, Hkv, D, W = case["Hq"], case["Hkv"], case["D"], case["window"]
    cache = build_cache(seq_lens, Hkv=Hkv, D=D, block_size=case["block"], seed=seed,
                        device=DEVICE, layout=case["layout"])
    q, qsl = make_queries(q_lens, Hq=Hq, D=D, seed=seed + 7, dtype=DTYPES[case["dtype"]],
                          device=DEVICE)
    T, R, q_max = sum(q_lens), len(q_lens), max(q_lens)
    cus = torch.cuda.get_device_properties(DEVICE).multi_processor_count
    s = {"case": case, "cache": cache, "q": q, "qsl": qsl, "out": torch.empty_like(q),
         "scale": 1.0 / math.sqrt(D), "none": torch.empty(0, device=DEVICE)}
    if case["one_launch"]:
        # The op itself, with a plan of the whole batch.
        ts = planner.workspace_token_splits(max_num_seqs=R, q_dec_max=1, Hkv=Hkv, D=D,
                                            num_sms=cus)
        plan = planner.plan_launch(num_tokens=T, num_reqs=R, max_query_len=q_max, G=Hq // Hkv,
                                   Hkv=Hkv, D=D, num_sms=cus, is_prefill=case["chunks"] > 0,
                                   ws_token_splits=max(ts, T), window=W)
        s.update(plan=plan, q_max=q_max, ws_o=s["none"], ws_lse=s["none"])
        if plan.num_splits > 1:
            s.update(ws_o=torch.empty(plan.ws_o_shape, device=DEVICE),
                     ws_lse=torch.empty(plan.ws_lse_shape, device=DEVICE))
        return s
    # The engine's forward: the step's slices, made once for all layers, and
    # the workspace, reserved once at load.
    builder = SliceBuilder(num_heads_q=Hq, num_kv_heads=Hkv, head_size=D, window=W,
                           max_num_seqs=MAX_NUM_SEQS, q_verify=case["q"], num_cus=cus,
                           device=DEVICE)
    step = builder.build(query_start_loc=qsl, query_start_loc_cpu=qsl.cpu(),
                         seq_lens=cache.seq_lens, block_table=cache.block_table, num_reqs=R,
                         num_actual_tokens=T, max_query_len=q_max, causal=case["causal"])
    used = max(p.plan.ws_token_splits_used for p in (step.decode, step.prefill) if p is not None)
    ws_o = torch.empty(used * Hq * D, device=DEVICE)
    ws_lse = torch.empty(used * Hq, device=DEVICE)
    s.update(step=step, reserved=builder.ws_token_splits, workspace=lambda o, lse: (
        ws_o[: math.prod(o)].view(o), ws_lse[: math.prod(lse)].view(lse)))
    return s


def _prepare_write(case, seed):
    T, Hq, Hkv, D = case["tokens"], case["Hq"], case["Hkv"], case["D"]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    # Keys and values as the fused projection leaves them, behind the queries.
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, generator=gen, device=DEVICE).to(
        DTYPES[case["dtype"]])
    key = qkv[:, Hq * D : (Hq + Hkv) * D].view(T, Hkv, D)
    value = qkv[:, (Hq + Hkv) * D :].view(T, Hkv, D)
    pages = -(-T // case["block"]) + 3
    storage = torch.zeros(pages * case["block"] * Hkv * cell_bytes(D), dtype=torch.int8,
                          device=DEVICE)
    views = carve_views(storage, num_blocks=pages, block_size=case["block"], Hkv=Hkv, D=D,
                        layout=case["layout"])
    ids = torch.randperm(pages, generator=gen, device=DEVICE)
    pos = torch.arange(T, device=DEVICE)
    slots = ids[pos // case["block"]] * case["block"] + pos % case["block"]
    return {"case": case, "key": key, "value": value, "views": views, "slots": slots,
            "storage": storage}


def run(s):
    case = s["case"]
    if case["kind"] == "write":
        ops.reshape_and_cache_int8(s["key"], s["value"], *s["views"], s["slots"])
        return s["storage"]
    c = s["cache"]
    views = (c.k_cache, c.v_cache, c.k_scale, c.v_scale)
    if case["one_launch"]:
        ops.pth_flash_attn_fwd(s["out"], s["q"], *views, c.block_table, c.seq_lens, s["qsl"],
                               s["q_max"], s["plan"].wm, s["plan"].num_splits, s["scale"],
                               s["ws_o"], s["ws_lse"], case["window"], case["causal"])
        return s["out"]
    return run_slices(s["step"], query=s["q"], output=s["out"], caches=views, scale=s["scale"],
                      window=case["window"], workspace=s["workspace"], no_workspace=s["none"],
                      reserved_token_splits=s["reserved"])


def tolerance(case):
    """Written cells are bytes. Attention rounds its output once to the query's
    type; two correct implementations lie a rounding of it apart."""
    if case["kind"] == "write":
        return "exact"
    return {"rel": 7e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 1e-3, "max": 4e-3}


def exact(case, seed):
    """Attention in 64 bits over the cells' own bytes."""
    if case["kind"] == "write":
        return None
    s = prepare(case, seed)
    q, storage, table = s["q"], s["cache"].storage, s["cache"].block_table
    Hq, Hkv, D, BS = case["Hq"], case["Hkv"], case["D"], case["block"]
    G, C = Hq // Hkv, 2 * D + 8
    cells = storage.view(-1, BS, Hkv, C) if case["layout"] == "NHD" else \
        storage.view(-1, Hkv, BS, C).transpose(1, 2)
    out, t0 = torch.empty(q.shape, dtype=torch.float64, device=q.device), 0
    for r, (n, L) in enumerate(zip(*lengths(case))):
        lo, hi = _visible(case, n, L)
        first, last = int(lo[0]) // BS, -(-int(hi[-1]) // BS)
        got = cells[table[r, first:last].long()].reshape(-1, Hkv, C)
        got = got[: int(hi[-1]) - first * BS].transpose(0, 1).contiguous()  # [Hkv, keys, C]
        scale = got.view(-1, C // 4, 4).contiguous().view(torch.float32).double()
        scale = scale.view(Hkv, -1, C // 4)
        k = got[..., :D].double() * scale[..., D // 4, None]
        v = got[..., D + 4 : 2 * D + 4].double() * scale[..., D // 2 + 1, None]
        pos = torch.arange(first * BS, int(hi[-1]), device=q.device)
        step = max(1, (1 << 28) // (Hq * len(pos)))
        lo_t, hi_t = (torch.from_numpy(x).to(q.device) for x in (lo, hi))
        for a in range(0, n, step):
            b = min(n, a + step)
            rows = q[t0 + a : t0 + b].double().view(b - a, Hkv, G, D).permute(1, 0, 2, 3)
            x = rows.reshape(Hkv, (b - a) * G, D) @ k.transpose(1, 2).contiguous()
            seen = (pos >= lo_t[a:b, None]) & (pos < hi_t[a:b, None])
            seen = seen.repeat_interleave(G, 0)
            p = torch.softmax((x * s["scale"]).masked_fill(~seen, -math.inf), -1)
            o = (p @ v).view(Hkv, b - a, G, D).permute(1, 0, 2, 3)
            out[t0 + a : t0 + b] = o.reshape(b - a, Hq, D)
        t0 += n
    return out
