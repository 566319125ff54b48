"""The combine's eight-columns-a-thread form (bf16 route rows of whole 16-byte pieces): the oracle's bits, with more ranks than
are requested at once, and beside the narrow form's at n that is no multiple of eight."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,top_k,n", [(1, 1, 8), (5, 11, 520), (512, 8, 1024), (3, 8, 516), (2, 16, 24)])
def test_combine_wide(ctx, orc, rows, top_k, n):
    import aq_mi355
    say("moe combine wide", rows, top_k, n)
    rng = np.random.default_rng(rows + n)
    yb = F.f32_to_bf16_bits(rng.normal(0, 1, (rows * top_k, n)).astype(np.float32))
    y = F.bf16_bits_to_f32(yb).reshape(rows * top_k, n)
    w = rng.uniform(-1, 1, rows * top_k).astype(np.float32)
    dw, dy, o32, o16 = ctx.to_device(w), ctx.to_device(yb), ctx.alloc(rows * n * 4), ctx.alloc(rows * n * 2)
    for steps in (False, True):
        flag = aq_mi355.AQ_BF16_STEPS if steps else 0
        want = orc.moe_combine(y, w, rows, top_k, n, bf16_steps=steps) if steps else orc.moe_combine(y, w, rows, top_k, n)
        ctx.moe_combine(dy, dw, o32, rows, top_k, n, aq_mi355.AQ_OUT_F32 | flag)
        ctx.moe_combine(dy, dw, o16, rows, top_k, n, flag)
        ctx.sync()
        assert np.array_equal(o32.download(np.float32, rows * n).reshape(rows, n), want.reshape(rows, n))
        assert np.array_equal(o16.download(np.uint16, rows * n).reshape(rows, n), F.f32_to_bf16_bits(want).reshape(rows, n))
    for t in (dw, dy, o32, o16):
        t.free()
