"""Softmax weights below float32's normal range are kept, wherever a decode makes one.

The dominant block's values are zero, so an output holds nothing but the contributions of the others, whose
weights beside it are 2^-127 to 2^-138: subnormal in float32, and lost if any weight on the way -- a chunk's, a
rescale's, a wave's, a workgroup's -- is flushed to zero."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dominant", [0, 1, 37, 79])  # ascending position among 80 blocks: every step, wave and workgroup sees it early or late
@pytest.mark.parametrize(("g", "d", "dt", "where", "q_f32"), [
    (4, 64, torch.float16, "pairs", False), (4, 128, torch.bfloat16, "pairs", False), (1, 64, torch.float16, "pairs", False), (8, 128, torch.bfloat16, "pairs", False),
    (4, 64, torch.float16, "records", False), (4, 128, torch.bfloat16, "records", False), (1, 64, torch.float16, "records", False), (8, 64, torch.float16, "records", False),
    (4, 64, torch.float16, "pairs", True), (2, 64, torch.float16, "records", True), (8, 64, torch.float16, "records", True), (4, 128, torch.bfloat16, "host", False),
])
def test_subnormal_weights_reach_the_output(g: int, d: int, dt: torch.dtype, where: str, q_f32: bool, dominant: int) -> None:
    from lazykv_amd import kernels
    from lazykv_amd.pinned import pinned_empty
    from lazykv_amd.quant import pack

    print(f"small weights: g={g} d={d} {dt} {where} q_f32={q_f32} dominant={dominant}", flush=True)
    h, bs, n = 2, 16, 80
    key = [0.0 if b == dominant else -(127.0 + b % 12) for b in range(n)]
    value = [0.0 if b == dominant else 2.0**15 * (1 + (b % 4) / 4) for b in range(n)]
    pool = torch.zeros((n, h, 2, bs, d), dtype=dt)  # one value per block: exact as a record too
    pool[:, :, 0, :, 0] = torch.tensor(key).to(dt)[:, None, None]
    pool[:, :, 1] = torch.tensor(value).to(dt)[:, None, None, None]
    if where == "records":
        store = pack(pool.cuda())
        sel = kernels.record_source(store, dt)
    else:
        store = pinned_empty(tuple(pool.shape), dt) if where == "host" else torch.empty_like(pool, device="cuda")
        store.copy_(pool)
        sel = kernels.pool_source(store)
    q = torch.zeros((h * g, d), dtype=torch.float32 if q_f32 else dt, device="cuda")
    q[:, 0] = 1.0
    idx = torch.arange(n, dtype=torch.int32, device="cuda").repeat(h, 1)
    out, lse = kernels.sparse_decode(q, n_kv=h, block_size=bs, scale=math.log(2.0), sel=sel, idx=idx, out_dtype=torch.float32)
    weight = np.exp(np.float64(np.float32(math.log(2.0))) * np.array(key))
    want = float((weight * np.array(value)).sum() / weight.sum())
    # A weight (or a factor of it: a chunk's, wave's or workgroup's) is rounded to a multiple of 2^-149, up to four times, and the
    # exponents, up to 138, carry a relative error of 2^-22.
    bound = 4 * 2.0**-150 * sum(value) + 138 * 2.0**-22 * want
    got = out.double().cpu().numpy()
    assert np.abs(got - want).max() < bound, (float(got.min()), float(got.max()), want)
    assert np.abs(lse.cpu().numpy() - math.log(bs)).max() < 1e-5
