"""The cache writer's two kernels (16-byte loads of aligned rows; one wave per
row otherwise) give the oracle's bytes: every head size and source type, part
filled work-groups, skipped tokens, padded token strides, both layouts, and
non-finite values, the same rows once on 16-byte addresses and once off them."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from test_writer import _cache, _expected, _write

pytestmark = pytest.mark.gpu


def _rows(x: torch.Tensor, off: int, pad: int) -> torch.Tensor:
    """x's values in a view `off` elements into its storage, tokens `pad` apart."""
    T, H, D = x.shape
    buf = torch.zeros(off + T * (H * D + pad), dtype=x.dtype, device=x.device)
    v = buf[off:].as_strided((T, H, D), (H * D + pad, D, 1), off)
    v.copy_(x)
    return v


@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_both_kernels(D, dtype, layout):
    for T, H, bs in [(1, 1, 16), (5, 3, 48), (67, 8, 16), (130, 5, 17)]:
        g = torch.Generator().manual_seed(D + T)
        key = torch.randn(T, H, D, generator=g).mul_(torch.rand(T, H, 1, generator=g) * 9).to(dtype)
        val = torch.randn(T, H, D, generator=g).to(dtype)
        val[0, 0] = 0.0  # the scale's floor
        nb = -(-T // bs) + 2
        slots = torch.randperm(nb * bs, generator=g)[:T].to(torch.int64)
        if T > 4:
            slots[3] = -1
            slots[4] = nb * bs  # out of the cache
        stored = []
        for off, pad in [(0, 0), (0, 16), (1, 0), (0, 1)]:
            st, views = _cache(nb, bs, H, D, "cuda", layout=layout)
            _write(_rows(key.cuda(), off, pad), _rows(val.cuda(), off, pad), views, slots.cuda())
            stored.append(st.cpu())
            kc, vc, ks, vs = (x.cpu().numpy() for x in views)
            for x, qc, sc in [(key, kc, ks), (val, vc, vs)]:
                q, s = _expected(x)
                for t in range(T):
                    at = int(slots[t])
                    if at < 0 or at >= nb * bs:
                        continue
                    assert np.array_equal(qc[at // bs, at % bs], q[t]), (T, off, pad, t)
                    assert np.array_equal(sc[at // bs, at % bs].view(np.int32), s[t].view(np.int32))
        for st in stored[1:]:  # skipped cells too
            assert torch.equal(st, stored[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_non_finite_values_alike(dtype):
    x = torch.randn(6, 2, 128, dtype=torch.float32)
    x[0, 0, 5], x[1, 1, 127], x[2, 0, 0], x[3, 1, 64:] = np.nan, np.inf, -np.inf, np.nan
    x = x.to(dtype).cuda()
    out = []
    for off in (0, 1):
        st, views = _cache(1, 16, 2, 128, "cuda")
        _write(_rows(x, off, 0), _rows(x, off, 0), views, torch.arange(6, device="cuda"))
        out.append(st.cpu())
    assert torch.equal(out[0], out[1])
