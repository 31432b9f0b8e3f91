"""The D = 64 unit kernels on paged cell caches (attn_paged64.hip) against the
fp64 oracle: whole slot rows of 8 KV heads and per-wave staging of any other
cell, at the edges of their 64-key steps, 32-key chunks and 16-key groups.

The gates are those of the register-load kernel, whose arithmetic they share
(test_attn_gpu.check_case).
"""

from __future__ import annotations

import pytest
import torch

from cases import Batch, Case, assert_parity, compare, materialize, oracle_of
from test_attn_gpu import check_case, last_kernel, run_capi, run_op

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 95, 96, 97, 127, 128, 129, 193, 1000]


def cases():
    for name, heads in [("rows", {"Hq": 32, "Hkv": 8}), ("rows-g1", {"Hq": 8, "Hkv": 8}),
                        ("staged", {"Hq": 16, "Hkv": 4}), ("staged-h9", {"Hq": 9, "Hkv": 9})]:
        heads = {**heads, "D": 64}
        R = len(EDGES)
        yield Case(f"p64-{name}-edges", q_lens=[1] * R, seq_lens=EDGES, seed=500, **heads)
        yield Case(f"p64-{name}-verify", q_lens=[3, 0, 4, 1, 4], seq_lens=[3, 9, 260, 700, 4099],
                   seed=501, **heads)
        yield Case(f"p64-{name}-fp16q", q_lens=[1, 2], seq_lens=[800, 77], q_dtype=torch.float16,
                   seed=502, **heads)
        yield Case(f"p64-{name}-hnd", q_lens=[1, 2], seq_lens=[900, 130], layout="HND", seed=503,
                   **heads)
        yield Case(f"p64-{name}-bs48", q_lens=[1, 1, 2], seq_lens=[500, 47, 1999], block_size=48,
                   seed=504, **heads)
        yield Case(f"p64-{name}-bs528-pad", q_lens=[2, 1], seq_lens=[1200, 300], block_size=528,
                   pad_tokens=3, pad_page_bytes=72, seed=505, **heads)
        yield Case(f"p64-{name}-many", q_lens=[1] * 70, seq_lens=[5 + 13 * i for i in range(70)],
                   seed=506, **heads)
    yield Case("p64-rows-g64", q_lens=[1, 1], seq_lens=[333, 90], Hq=128, Hkv=2, D=64, seed=507)


@pytest.mark.parametrize("S", [1, 2, 5])
@pytest.mark.parametrize("case", list(cases()), ids=lambda c: c.name)
def test_paged64(case, S):
    check_case(case, num_splits=S)
    # Whole slot rows: NHD cells of 8 KV heads, at most 16 rows a tile.
    rows = case.layout == "NHD" and case.Hkv == 8 and max(case.q_lens) * case.G <= 16
    kernel = "attn_fwd_pagerows64" if rows else "attn_fwd_staged64"
    if case.G == 64 and S == 1:  # a request's 64 rows reach the wide-block kernel's line
        kernel = "attn_fwd_wide"
    assert last_kernel() == kernel


def test_paged64_repeats():
    """The op's launch, equal bit for bit over repeats (the page-row kernel's
    shared steps hold no race)."""
    c = Case("p64-repeat", q_lens=[1] * 6, seq_lens=[9000, 64, 4000, 1, 8191, 333], Hq=32, Hkv=8,
             D=64, seed=510)
    b = materialize(c, "cuda")
    first = run_op(b)
    assert last_kernel() == "attn_fwd_pagerows64"
    for _ in range(5):
        assert torch.equal(run_op(b).view(torch.int16), first.view(torch.int16))


@pytest.mark.parametrize("S", [1, 3])
@pytest.mark.parametrize("D,kernel", [(64, "attn_fwd_staged64"), (128, "attn_fwd_staged")])
def test_overlapping_streams(D, kernel, S):
    """K as V in cells of the page-row size: no stream ends with the cell, so the
    rest of the last one may be nobody's memory and whole rows are not loaded."""
    c = Case(f"p64-k-as-v-d{D}", q_lens=[1, 2], seq_lens=[300, 77], Hq=32, Hkv=8, D=D, seed=511)
    b = materialize(c, "cuda")
    host = b.cache.to("cpu")
    host.v_cache.copy_(host.k_cache)
    host.v_scale.copy_(host.k_scale)
    ref, ref_lse, valid = oracle_of(Batch(c, host, b.q.cpu(), b.qsl.cpu()))
    b.cache.v_cache, b.cache.v_scale = b.cache.k_cache, b.cache.k_scale
    out, lse = run_capi(b, num_splits=S)
    assert last_kernel() == kernel
    assert_parity(compare(out, lse, ref, ref_lse, valid), name=c.name, strict=False)
