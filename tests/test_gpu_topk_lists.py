"""The k largest packed values by way of lists: lists of exactly as many entries as are read together, hold, or overflow; as many
lists as one form of the merge takes and one more; a last list of one entry."""
import numpy as np
import pytest

from gpu_util import say
from test_gpu_head import _u64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [64 * 256, 64 * 1024 + 1, 64 * 4096, 64 * 4096 + 1])
@pytest.mark.parametrize("top_k", [40, 64])
@pytest.mark.parametrize("planted", [1, 64, 65, 128, 129])
def test_lists(ctx, count, top_k, planted):
    say("packed topk lists", count, top_k, planted)
    rng = np.random.default_rng(count + top_k + planted)
    packed = rng.integers(1 << 40, 1 << 62, count, dtype=np.uint64)
    packed[512:512 + planted] = (np.uint64(0xF0000000) << np.uint64(32)) | rng.permutation(1 << 20)[:planted].astype(np.uint64)
    packed[-1] = np.uint64(0xF1) << np.uint64(56)
    din, dout = ctx.to_device(packed), ctx.to_device(np.full(top_k, 0xDEADBEEF, np.uint64))
    ctx.packed_topk(din, count, top_k, dout)
    ctx.sync()
    assert np.array_equal(_u64(dout, top_k), np.sort(packed)[::-1][:top_k])
    din.free()
    dout.free()


@pytest.mark.parametrize("count,top_k", [(6000, 40), (6000, 64), (64 * 1024, 1), (64 * 4096 + 1, 64)])
@pytest.mark.parametrize("step", [1, 1 << 9, 1 << 14])
def test_scores_that_agree_in_their_high_bits(ctx, count, top_k, step):
    """... and differ in the last ones, or are a few values many times over."""
    say("packed topk, close scores", count, top_k, step)
    rng = np.random.default_rng(count + top_k + step)
    near = (np.float32(1000) + rng.standard_normal(count).astype(np.float32) * np.float32(0.3)).view(np.uint32)
    key = near // np.uint32(step) * np.uint32(step) | np.uint32(0x80000000)
    packed = (key.astype(np.uint64) << np.uint64(32)) | np.arange(count, dtype=np.uint64)
    din, dout = ctx.to_device(packed), ctx.to_device(np.full(top_k, 0xDEADBEEF, np.uint64))
    ctx.packed_topk(din, count, top_k, dout)
    ctx.sync()
    assert np.array_equal(_u64(dout, top_k), np.sort(packed)[::-1][:top_k])
    din.free()
    dout.free()
