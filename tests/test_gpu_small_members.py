"""Matrices of up to 528 rows in whole sets of 16 on the token tiles: k and v beside q in one grid with the bytes of their own calls, at
the numbers of rows of x where a call changes form; groups of 128 from two rows on (4 bit, K a multiple of 512), of 32 from three."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,gs,M,K,Ns", [(4, 64, 9, 1216, (1040, 448, 528)), (4, 64, 32, 832, (640, 16, 512)), (4, 64, 33, 2048, (2064, 512, 256)),
                                            (8, 64, 64, 1216, (1536, 448, 448)), (4, 32, 48, 960, (600, 256, 528)), (8, 32, 40, 512, (544, 512, 512)),
                                            (4, 128, 2, 1536, (1536, 384, 32)), (8, 128, 5, 896, (1024, 256, 7)), (4, 128, 64, 384, (531, 512, 272)),
                                            (4, 32, 3, 1216, (1537, 448, 33))])
def test_members_beside_a_wide_matrix(ctx, bits, gs, M, K, Ns):
    import aq_mi355
    say("small members", bits, gs, M, K, Ns)
    x = F.synthetic_x(M, K, seed=3300)
    dx, f32 = ctx.to_device(x), aq_mi355.AQ_OUT_F32
    mats = [F.synthetic_affine(n, K, bits, gs, seed=3301 + i) for i, n in enumerate(Ns)]
    dws = [DeviceAffine(ctx, *m) for m in mats]
    one, ys = ctx.alloc(M * max(Ns) * 4), [ctx.alloc(M * n * 4) for n in Ns]
    ctx.qmv_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, bits, f32)
    ctx.sync()
    for m, d, n, y in zip(mats, dws, Ns, ys):
        got = y.download(np.float32, M * n)
        ctx.qmv(dx, d.w, d.s, d.b, one, M, K, n, gs, bits, f32)
        ctx.sync()
        assert ctx.last_variant(0).startswith("qmvt_"), (n, ctx.last_variant(0))
        assert np.array_equal(got.view(np.uint32), one.download(np.uint32, M * n)), "member of %d rows" % n
        check_accumulators(got.reshape(M, n), F.reference_f64(x, *m, bits, gs, K), "member of %d rows" % n)
    for t in [dx, one] + ys + dws:
        t.free()
