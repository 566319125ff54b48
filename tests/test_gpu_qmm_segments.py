"""The fp16-operand matmul kernels where scales and biases pass through LDS in segments: K that ends in a segment's first or last quad,
rows of scales at any even address, arrays of scales shorter than one load, every tile."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, run_qmv, say

pytestmark = pytest.mark.gpu


# a segment is 8 or 16 elements of a row, 4 / gs_blocks of them (groups of 32: 8) a quad of four 64-code blocks.  Ends: one block, a
# whole segment, one block into the next, the middle of a quad of the third; fewer than eight scales in all
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("gs,M,K,N", [(32, 33, 64, 3), (32, 97, 512, 67), (32, 40, 832, 131), (32, 300, 1984, 131), (64, 65, 64, 5), (64, 97, 1024, 67), (64, 40, 1088, 131),
                                      (64, 130, 2240, 35), (128, 33, 128, 1), (128, 97, 2048, 67), (128, 40, 2176, 35)])
def test_every_tile_over_segments_of_scales(ctx, bits, gs, M, K, N):
    import aq_mi355
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=4100 + K)
    x = F.synthetic_x(M, K, seed=4101 + M)
    dw = DeviceAffine(ctx, words, s, b)
    ref, first = F.reference_f64(x, words, s, b, bits, gs, K), None
    prefix = "qmmh_" if bits == 4 else "qmmh8_"
    # (the rule's tile too: groups of 32 have its shares of K on every tile)
    tiles = [(i, n) for i, n in enumerate(aq_mi355.variant_names(1)) if n.startswith(prefix)] + ([(-1, prefix)] if gs == 32 else [])
    for i, name in tiles:
        say("segments", name, gs, M, K, N)
        ctx.force_variant(1, i)
        try:
            acc = run_qmv(ctx, x, dw, M, K, N, gs, bits, True, fn="qmm")
            assert ctx.last_variant(1).startswith(name)
        finally:
            ctx.force_variant(1, -1)
        check_accumulators(acc, ref, name)
        first = acc if first is None else first
        assert np.array_equal(acc.view(np.uint32), first.view(np.uint32)), name
    assert first is not None
    dw.free()
