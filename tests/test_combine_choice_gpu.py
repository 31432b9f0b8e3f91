"""The op's combine on either side of the request count up to which a row's
splits are shared by the waves of a work-group: launches whose split bound is
far above 64, with rows of one live split, of few, and of more than a block of
64 (one long request among short ones), against the fp64 oracle."""

from __future__ import annotations

import pytest
import torch

from cases import Case, assert_parity, compare, materialize, oracle_of
from test_attn_gpu import run_capi, run_op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("R", [16, 17, 31])
@pytest.mark.parametrize("long", [200, 30000])
def test_combine_choice(D, R, long):
    c = Case(f"combine-d{D}-r{R}-{long}", q_lens=[1] * R, seq_lens=[40 + 7 * i for i in range(R - 1)] + [long],
             Hq=16, Hkv=4, D=D, seed=600 + R)
    assert c.plan().num_splits > 64
    b = materialize(c, "cuda")
    out = run_op(b)
    ref, _, valid = oracle_of(b, threads=16)
    assert_parity(compare(out, None, ref, None, valid), name=c.name, strict=False)
    assert torch.equal(run_op(b).view(torch.int16), out.view(torch.int16))


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("chunks", [64, 65, 66, 127, 128, 129, 255, 256, 257, 262, 938])
def test_long_row_among_short_ones(D, chunks):
    """A row of exactly `chunks` live splits (one KV head: every chunk of a launch
    this small is a split) beside rows of two, on the kernel that cuts a long
    row into runs: one block, the last wave's run short or empty, runs of more
    than a block; output and LSE."""
    c = Case(f"combine-row-d{D}-{chunks}", q_lens=[1] * 17,
             seq_lens=[40] * 8 + [32 * chunks - 5] + [60] * 8, Hq=4, Hkv=1, D=D, seed=620)
    assert c.plan().num_splits > chunks
    b = materialize(c, "cuda")
    ref, ref_lse, valid = oracle_of(b, threads=16)
    out, lse = run_capi(b, out_dtype=torch.float32)
    res = compare(out, lse, ref, ref_lse, valid)
    assert res["finite"] and res["max_abs"] <= 1e-4 and res["lse_max_abs"] <= 1e-3, res
