"""The wide-block kernel (attn_wide.hip) against the fp64 oracle: prefill
launches with split partials at every head size, and single-split ones at
D = 64 and 256, at the edges of its blocks, steps and score tiles.

The gates are those of the unit kernels (test_attn_gpu.check_case): the
output within the parity tolerance beyond its storage rounding, and the
fp32-output launch within 1e-4 (P is a bf16 hi + lo pair, as there).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from cases import Batch, Case, abs_v_batch, assert_parity, compare, materialize, oracle_of
from test_attn_gpu import check_case, last_kernel, run_capi, run_op

pytestmark = pytest.mark.gpu


WIDE = "attn_fwd_wide"


def min_rows(D: int, S: int) -> int:
    """Mean query rows per request of the launcher's line (attn_launch.hip)."""
    if S == 1:
        return 384 if D == 256 else 64  # at D = 256 of at least 80 tokens
    return 3072 if D == 256 else 1280


# At D = 128 a launch needs 40 blocks of 256 rows as well at these lengths.
HEADS = {64: {"Hq": 8, "Hkv": 2, "D": 64}, 128: {"Hq": 32, "Hkv": 8, "D": 128},
         256: {"Hq": 8, "Hkv": 2, "D": 256}}


def cases():
    for D in (64, 128, 256):
        blk = 128 if D == 256 else 256  # rows of a block
        step = 32 if D == 256 else 64  # keys of a step
        m = min_rows(D, 2) // 4  # tokens of a request at four query heads per KV head
        heads = HEADS[D]
        # One block less, just, and more than full; keys at the step's edges.
        for i, (rows, keys) in enumerate([(blk - 4, 0), (blk, 1), (blk + 4, step - 1), (3 * blk, 17)]):
            q = m + rows // 4
            yield Case(f"wide-d{D}-rows{rows}", q_lens=[q], seq_lens=[-(-q // step) * step + step + keys],
                       seed=400 + i, **heads)
        yield Case(f"wide-d{D}-first", q_lens=[m + 3], seq_lens=[m + 3], seed=409, **heads)
        yield Case(f"wide-d{D}-ragged", q_lens=[m + 37, 0, 4 * m + 130, 1, m + 66, 40],
                   seq_lens=[m + 37, 9, 4 * m + 1500, 700, m + 67, 3000], seed=410, **heads)
        yield Case(f"wide-d{D}-fp16q-hnd", q_lens=[2 * m, 33], seq_lens=[2 * m + 800, 47], layout="HND",
                   q_dtype=torch.float16, seed=411, **heads)
        yield Case(f"wide-d{D}-bs48", q_lens=[m + 90, m], seq_lens=[m + 500, m + 1999], block_size=48,
                   seed=412, Hq=12, Hkv=2, D=D)
        yield Case(f"wide-d{D}-bs528-pad", q_lens=[m + 70, m + 41], seq_lens=[m + 1200, m + 300],
                   block_size=528, pad_tokens=3, pad_page_bytes=72, seed=413, **heads)
        t = 78 if D == 256 else m // 16  # one split at D = 256: 80 tokens
        yield Case(f"wide-d{D}-g64", q_lens=[t + 5, t + 3], seq_lens=[333, 90], Hq=64,
                   Hkv=1, D=D, seed=414) if D != 128 else \
            Case("wide-d128-g64", q_lens=[25, 23], seq_lens=[333, 90], Hq=192, Hkv=3, seed=414)
        yield Case(f"wide-d{D}-g1", q_lens=[4 * m + 300, 4 * m + 70], seq_lens=[4 * m + 300, 4 * m + 500],
                   Hq=4 if D == 128 else 2, Hkv=4 if D == 128 else 2, D=D, seed=415)
        yield Case(f"wide-d{D}-many", q_lens=[m // 16 + i % 9 for i in range(70)],
                   seq_lens=[m // 16 + 9 + 3 * i for i in range(70)], seed=416, Hq=64, Hkv=1, D=D)
    heads = HEADS[128]
    yield Case("wide-window", q_lens=[500, 400], seq_lens=[1200, 3000], window=64, seed=420, **heads)
    yield Case("wide-window-odd", q_lens=[531, 133], seq_lens=[2000, 800], window=333, seed=421, **heads)
    yield Case("wide-noncausal", q_lens=[600, 130], seq_lens=[900, 150], causal=False, seed=422, **heads)
    yield Case("wide-window-noncausal", q_lens=[480, 330], seq_lens=[2000, 400], window=100,
               causal=False, seed=423, **heads)


@pytest.mark.parametrize("S", [1, 2, 5])
@pytest.mark.parametrize("case", list(cases()), ids=lambda c: c.name)
def test_wide(case, S):
    if S == 1 and case.D == 128:
        pytest.skip("the row-block kernel's launch")
    if S == 1 and case.D == 256 and case.T < 80 * len(case.q_lens):
        pytest.skip("the unit kernels' launch")
    check_case(case, num_splits=S)
    assert last_kernel() == WIDE


@pytest.mark.parametrize("D", [64, 128, 256])
def test_wide_op_and_repeats(D):
    """The op's launch (attention + combine) at the planner's split count, equal
    bit for bit over repeats."""
    c = Case(f"wide-op-d{D}", q_lens=[1000, 600], seq_lens=[2000, 633], Hq=8, Hkv=2, D=D, seed=430)
    assert c.plan().num_splits > 1
    b = materialize(c, "cuda")
    first = run_op(b)
    assert last_kernel() == WIDE
    ref, _, valid = oracle_of(b, threads=16)
    assert_parity(compare(first, None, ref, None, valid), name=c.name, strict=False)
    for _ in range(5):
        assert torch.equal(run_op(b).view(torch.int16), first.view(torch.int16))


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("big", [2.0 ** 3, 2.0 ** 6, 2.0 ** 12, 2.0 ** 40])
def test_wide_large_v_scales(D, big):
    """V scales that grow mid-stream by factors far beyond fp16's range, of keys
    that some rows see, that are masked for others, or that weigh nothing in
    them: the small ones lose no bits. Checked relative to each row's largest
    output: a term lies within 2^-17 = 7.6e-6 of itself, and the errors of a
    row's terms are as good as independent."""
    c = Case(f"wide-bigv-d{D}", q_lens=[800, 770], seq_lens=[800, 990], D=D, Hq=8, Hkv=2, seed=440)
    b = materialize(c, "cuda")
    ch, bt = b.cache, b.cache.block_table.cpu()
    for r, (lo, hi, f) in enumerate([(100, 200, big), (400, 410, big * big)]):
        for t in range(lo, min(hi, c.seq_lens[r])):
            ch.v_scale[int(bt[r, t // c.block_size]), t % c.block_size] *= f
    torch.cuda.synchronize()
    ref_out, ref_lse, valid = oracle_of(b)
    out, lse = run_capi(b, num_splits=3, out_dtype=torch.float32)
    assert last_kernel() == WIDE
    o, r = out.cpu().numpy()[valid].astype(np.float64), ref_out[valid]
    assert np.isfinite(o).all()
    rel = np.abs(o - r) / np.abs(r).max(axis=-1, keepdims=True)
    print(f"large V scales d{D} {big:g}: worst {rel.max():.3g}")
    assert rel.max() <= 1e-5, rel.max()
    assert np.abs(lse.cpu().numpy()[valid] - ref_lse[valid]).max() <= 1e-3


# ------------------------------------------------- weights far below the largest
# The kernel's numerics are those of the unit kernels: P is a hi + lo pair of 16
# significant bits at any size, so a term p_i v_i of a row's sum is within
# 2^-17 of itself, and the scores, exponentials and fp32 sums add less than as
# much again: the oracle on |V| gives sum_i p_i |v_i| / l, and every output
# element lies within 2^-16 of that.
P_PAIR_UNIT = 2.0 ** -16
KEYS = 4096


def _sink(n, step, x, r):
    """Key 0 is 2^x above the rest, its V scale r times theirs."""
    score, vs = np.zeros(n), np.ones(n)
    score[0], vs[0] = x, r
    return score, vs


def _jump(n, step, x, r):
    """One step of equal keys, then one key 2^x above them, nothing after it."""
    score, vs = np.full(n, -80.0), np.ones(n)
    score[:step], score[step], vs[step] = 0.0, x, r
    return score, vs


def _tail(n, step, x, r):
    """Key 0 over a long tail 2^x below it, and a key of no weight whose V scale
    is 1 / r times theirs."""
    score, vs = np.full(n, -x), np.ones(n)
    score[0], score[1], vs[1] = 0.0, -80.0, 1.0 / r
    return score, vs


def _small_weight_case(D, S):
    return Case(f"wide-small-d{D}", q_lens=[min_rows(D, 2) // 4 + 9], seq_lens=[KEYS], seed=450,
                **HEADS[D])


def _places(b, r, n):
    t = torch.arange(n, device="cuda")
    return b.cache.block_table[r, t // b.case.block_size].long(), t % b.case.block_size


@pytest.mark.parametrize("ratio", [1.0, 1 / 8, 1 / 100, 1 / 300])
@pytest.mark.parametrize("x", [17.5, 22.6, 25.0, 30.0])
@pytest.mark.parametrize("profile", [_sink, _jump, _tail], ids=lambda f: f.__name__[1:])
@pytest.mark.parametrize("D,S", [(64, 1), (64, 2), (128, 2), (256, 1), (256, 2)])
def test_wide_small_weights(D, S, profile, x, ratio):
    c = _small_weight_case(D, S)
    b = materialize(c, "cuda")
    b.q.fill_(1.0)
    score, vs = profile(KEYS, 32 if D == 256 else 64, x, ratio)
    pages, slots = _places(b, 0, KEYS)
    ch = b.cache
    ch.k_cache[pages, slots] = 1  # score = sqrt(D) k_scale
    f32 = {"dtype": torch.float32, "device": "cuda"}
    ch.k_scale[pages, slots] = torch.tensor(score * np.log(2) / np.sqrt(D), **f32)[:, None]
    ch.v_scale[pages, slots] = torch.tensor(0.01 * vs, **f32)[:, None]
    torch.cuda.synchronize()
    # All rows have one query: the oracle on the last token's, which sees every key.
    last = Case(c.name, q_lens=[1], seq_lens=[KEYS], **HEADS[D])
    lb = Batch(last, ch, b.q[-1:], torch.tensor([0, 1], dtype=torch.int32, device="cuda"))
    ref_out, ref_lse, _ = oracle_of(lb, threads=16)
    abs_out, _, _ = oracle_of(abs_v_batch(lb), threads=16)
    out, lse = run_capi(b, num_splits=S, out_dtype=torch.float32)
    assert last_kernel() == WIDE
    err = np.abs(out[-1:].cpu().numpy().astype(np.float64) - ref_out)
    worst = float((err / abs_out).max())
    print(f"d{D} S{S} {profile.__name__} x={x} ratio={ratio:.4f}: worst error / sum p|v| {worst:.3g}")
    assert worst <= P_PAIR_UNIT, worst
    assert np.abs(lse[-1:].cpu().numpy() - ref_lse).max() <= 1e-3


# ------------------------------------------------------------- non-finite inputs
def _sees(c, r, key):
    """Rows (tokens of the batch) that see position `key` of request r."""
    seen = np.zeros(c.T, bool)
    t0, n, L = sum(c.q_lens[:r]), c.q_lens[r], c.seq_lens[r]
    p = np.arange(L - n, L)
    seen[t0:t0 + n] = (p >= key) & ((c.window == 0) | (key >= p - c.window + 1))
    return torch.from_numpy(seen).cuda()


@pytest.mark.parametrize("stream", ["k_scale", "v_scale"])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("D,S,window", [(64, 1, 0), (64, 2, 0), (128, 2, 0), (128, 2, 150), (256, 1, 0),
                                        (256, 3, 0)])
def test_wide_non_finite_scale(D, S, window, bad, stream):
    """A non-finite scale reaches the rows that see its key, and no other row of
    the block; a V scale never reaches a row's LSE."""
    m = min_rows(D, 2) // 4
    c = Case(f"wide-nonfinite-d{D}", q_lens=[m + 70, m], seq_lens=[m + 300, m + 41],
             window=window, seed=460, **HEADS[D])
    b = materialize(c, "cuda")
    clean, clean_lse = run_capi(b, num_splits=S, out_dtype=torch.float32)
    assert last_kernel() == WIDE
    key = c.seq_lens[0] - c.q_lens[0] + 133  # within a block's tokens
    pages, slots = _places(b, 0, c.seq_lens[0])
    getattr(b.cache, stream)[pages[key], slots[key]] = bad
    out, lse = run_capi(b, num_splits=S, out_dtype=torch.float32)
    seen = _sees(c, 0, key)
    assert 0 < int(seen.sum()) < c.q_lens[0]
    assert torch.equal(out[~seen].view(torch.int32), clean[~seen].view(torch.int32))
    assert torch.equal(lse[~seen].view(torch.int32), clean_lse[~seen].view(torch.int32))
    if stream == "v_scale":
        assert not torch.isfinite(out[seen]).any()
        assert torch.equal(lse.view(torch.int32), clean_lse.view(torch.int32))


@pytest.mark.parametrize("D,S", [(64, 1), (128, 2), (256, 1)])
def test_wide_infinite_query(D, S):
    """A row whose fp16 query holds an infinity is NaN whatever the sign of the
    keys' bytes there (0 where it is split: a split without a sum is no split to
    the combine), and no other row changes."""
    m = min_rows(D, 2) // 4
    c = Case(f"wide-infq-d{D}", q_lens=[m + 33] * 12, seq_lens=[m + 90] * 12, D=D, Hq=8, Hkv=2,
             q_dtype=torch.float16, seed=470)
    b = materialize(c, "cuda")
    b.cache.k_cache[..., 5] = -7
    clean, _ = run_capi(b, num_splits=S, out_dtype=torch.float32)
    assert last_kernel() == WIDE
    rows = torch.tensor([(m + 33) * r + 7 + 23 * r for r in range(12)], device="cuda")
    heads = torch.arange(12, device="cuda") % 8
    b.q[rows, heads, 5] = float("inf")
    out, _ = run_capi(b, num_splits=S, out_dtype=torch.float32)
    bad = out[rows, heads]
    nan = torch.isnan(bad).all(-1)
    assert nan.any() if S > 1 else nan.all()
    assert (nan | (bad == 0).all(-1)).all()
    out[rows, heads] = clean[rows, heads]
    assert torch.equal(out.view(torch.int32), clean.view(torch.int32))


@pytest.mark.parametrize("D,S,heads,q_lens,kernel", [
    (64, 1, (8, 2), [16, 16], WIDE),
    (64, 1, (8, 2), [16, 15], "attn_fwd_staged64"),
    (256, 1, (12, 2), [80, 80], WIDE),
    (256, 1, (12, 2), [80, 79], "attn_fwd_paged256"),
    (256, 1, (8, 2), [96, 95], "attn_fwd_paged256"),
    (256, 1, (64, 1), [79], "attn_fwd_paged256"),
    (64, 4, (8, 1), [160], WIDE),
    (64, 4, (8, 1), [159], "attn_fwd_staged64"),
    (256, 4, (6, 1), [512], WIDE),
    (256, 4, (6, 1), [511], "attn_fwd_paged256"),
    (128, 4, (32, 4), [160, 160], WIDE),
    (128, 4, (32, 4), [160, 159], "attn_fwd_staged"),
    (128, 4, (32, 4), [202], "attn_fwd_staged"),  # 1,616 rows x 6,464 of all heads < 1,280 x 8,192
    (128, 4, (32, 4), [203], WIDE),
    (128, 4, (8, 1), [404], "attn_fwd_staged"),
    (128, 4, (8, 1), [405], WIDE),
])
def test_launch_lines(D, S, heads, q_lens, kernel):
    """Either side of the launcher's lines; the kernels agree at the parity gate."""
    c = Case(f"line-d{D}", q_lens=q_lens, seq_lens=[q + 50 for q in q_lens], Hq=heads[0],
             Hkv=heads[1], D=D, is_prefill=True, seed=480)
    check_case(c, num_splits=S)
    assert last_kernel() == kernel
