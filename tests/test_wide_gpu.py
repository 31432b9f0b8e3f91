"""The wide-block kernel (attn_wide.hip) against the fp64 oracle: prefill
launches with split partials at every head size, and single-split ones at
D = 64 and 256, at the edges of its blocks, steps and score tiles.

The gates are those of the unit kernels (test_attn_gpu.check_case): the
output within the parity tolerance beyond its storage rounding, and the
fp32-output launch within 1e-4. P is an fp16 hi + lo pair (22 significant
bits), so the arithmetic error is that of the fp32 sums.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from cases import Case, assert_parity, compare, materialize, oracle_of, tile_tokens
from test_attn_gpu import check_case, run_capi, run_op

pytestmark = pytest.mark.gpu


def wide(c: Case, S: int) -> bool:
    """The launcher's rule (attn_launch.hip)."""
    plan = c.plan()
    bq = tile_tokens(plan.wm, c.G, max(c.q_lens))
    return (c.block_size % 16 == 0 and bq * c.G > 32 and (S > 1 or c.D != 128)
            and c.T * c.G > 64 * len(c.q_lens))


def cases():
    for D in (64, 128, 256):
        blk = 128 if D == 256 else 256  # rows of a block
        step = 32 if D == 256 else 64  # keys of a step
        heads = {"Hq": 8, "Hkv": 2, "D": D}
        # One block less, just, and more than full; keys at the step's edges.
        for i, (rows, keys) in enumerate([(blk - 4, step), (blk, step + 1), (blk + 4, 2 * step - 1),
                                          (3 * blk, 16 * step + 17)]):
            q = rows // 4
            yield Case(f"wide-d{D}-rows{rows}", q_lens=[q], seq_lens=[max(q, keys)], seed=400 + i,
                       **heads)
        yield Case(f"wide-d{D}-ragged", q_lens=[37, 0, 130, 1, 66, 40], seq_lens=[37, 9, 1500, 700, 67, 3000],
                   seed=410, **heads)
        yield Case(f"wide-d{D}-fp16q-hnd", q_lens=[100, 33], seq_lens=[900, 47], layout="HND",
                   q_dtype=torch.float16, seed=411, **heads)
        yield Case(f"wide-d{D}-bs48", q_lens=[90, 50], seq_lens=[500, 1999], block_size=48, seed=412,
                   Hq=12, Hkv=2, D=D)
        yield Case(f"wide-d{D}-bs528-pad", q_lens=[70, 41], seq_lens=[1200, 300], block_size=528,
                   pad_tokens=3, pad_page_bytes=72, seed=413, **heads)
        yield Case(f"wide-d{D}-g64", q_lens=[5, 3], seq_lens=[333, 90], Hq=64, Hkv=1, D=D, seed=414)
        yield Case(f"wide-d{D}-g1", q_lens=[300, 70], seq_lens=[300, 2000], Hq=3, Hkv=3, D=D, seed=415)
        yield Case(f"wide-d{D}-many", q_lens=[20 + i % 9 for i in range(70)],
                   seq_lens=[40 + 13 * i for i in range(70)], seed=416, **heads)
    heads = {"Hq": 8, "Hkv": 2}
    yield Case("wide-window", q_lens=[200, 40], seq_lens=[900, 3000], window=64, seed=420, **heads)
    yield Case("wide-window-odd", q_lens=[131, 33], seq_lens=[2000, 800], window=333, seed=421, **heads)
    yield Case("wide-noncausal", q_lens=[100, 30], seq_lens=[400, 50], causal=False, seed=422, **heads)
    yield Case("wide-window-noncausal", q_lens=[80, 30], seq_lens=[2000, 300], window=100,
               causal=False, seed=423, **heads)


@pytest.mark.parametrize("S", [1, 2, 5])
@pytest.mark.parametrize("case", list(cases()), ids=lambda c: c.name)
def test_wide(case, S):
    if S == 1 and case.D == 128:
        pytest.skip("the row-block kernel's launch")
    assert wide(case, S), case.name
    check_case(case, num_splits=S)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_wide_op_and_repeats(D):
    """The op's launch (attention + combine) at the planner's split count, equal
    bit for bit over repeats."""
    c = Case(f"wide-op-d{D}", q_lens=[150, 70], seq_lens=[2000, 333], Hq=8, Hkv=2, D=D, seed=430)
    assert c.plan().num_splits > 1 and wide(c, c.plan().num_splits)
    b = materialize(c, "cuda")
    first = run_op(b)
    ref, _, valid = oracle_of(b, threads=16)
    assert_parity(compare(first, None, ref, None, valid), name=c.name, strict=False)
    for _ in range(5):
        assert torch.equal(run_op(b).view(torch.int16), first.view(torch.int16))


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("big", [2.0 ** 12, 2.0 ** 40])
def test_wide_large_v_scales(D, big):
    """V scales far beyond fp16's range that grow mid-stream: the growth
    threshold follows their exponent, so P V stays in range and rows that
    grow rescale what they hold. Checked relative to each row's largest
    output: every step is fp32 or 22 bits, so 1e-5 leaves a decade."""
    c = Case(f"wide-bigv-d{D}", q_lens=[96, 70], seq_lens=[300, 620], D=D, seed=440)
    assert wide(c, 3)
    b = materialize(c, "cuda")
    ch, bt = b.cache, b.cache.block_table.cpu()
    for r, (lo, hi, f) in enumerate([(100, 200, big), (400, 410, big * big)]):
        for t in range(lo, min(hi, c.seq_lens[r])):
            ch.v_scale[int(bt[r, t // c.block_size]), t % c.block_size] *= f
    torch.cuda.synchronize()
    ref_out, ref_lse, valid = oracle_of(b)
    out, lse = run_capi(b, num_splits=3, out_dtype=torch.float32)
    o, r = out.cpu().numpy()[valid].astype(np.float64), ref_out[valid]
    assert np.isfinite(o).all()
    rel = np.abs(o - r) / np.abs(r).max(axis=-1, keepdims=True)
    assert rel.max() <= 1e-5, rel.max()
    assert np.abs(lse.cpu().numpy()[valid] - ref_lse[valid]).max() <= 1e-3
