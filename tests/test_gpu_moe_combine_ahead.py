"""The combine's wide form at every number of ranks around those it requests at once (2, 4, 8): the oracle's bits, signed zeros,
infinities and NaN among the rows."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top_k", [1, 2, 3, 4, 5, 7, 8, 9, 17])
def test_ranks_requested_together(ctx, orc, top_k):
    import aq_mi355
    rows, n = 3, 520
    say("moe combine", rows, top_k, n)
    rng = np.random.default_rng(100 + top_k)
    y = rng.normal(0, 1, (rows * top_k, n)).astype(np.float32)
    y[:, :8] = -0.0
    y[0, 8], y[-1, 9], y[top_k, 10] = np.inf, -np.inf, np.nan
    yb = F.f32_to_bf16_bits(y)
    y = F.bf16_bits_to_f32(yb).reshape(rows * top_k, n)
    w = rng.uniform(0.01, 1, rows * top_k).astype(np.float32)
    dw, dy, o32, o16 = ctx.to_device(w), ctx.to_device(yb), ctx.alloc(rows * n * 4), ctx.alloc(rows * n * 2)
    for steps in (False, True):
        flag = aq_mi355.AQ_BF16_STEPS if steps else 0
        want = orc.moe_combine(y, w, rows, top_k, n, bf16_steps=steps).reshape(rows, n)
        ctx.moe_combine(dy, dw, o32, rows, top_k, n, aq_mi355.AQ_OUT_F32 | flag)
        ctx.moe_combine(dy, dw, o16, rows, top_k, n, flag)
        ctx.sync()
        got32, got16 = o32.download(np.uint32, rows * n).reshape(rows, n), o16.download(np.uint16, rows * n).reshape(rows, n)
        nan = np.isnan(want)  # (whose payload and sign are the machine's)
        assert nan.any() and np.array_equal(nan, np.isnan(got32.view(np.float32)))
        assert np.array_equal(got32[~nan], want.view(np.uint32)[~nan])
        assert np.array_equal(got16[~nan], F.f32_to_bf16_bits(want).reshape(rows, n)[~nan])
        assert np.isnan(F.bf16_bits_to_f32(got16)[nan]).all()
    for t in (dw, dy, o32, o16):
        t.free()
