"""Five to eight rows of x through several matrices in one grid and through a gated pair: every member has the bytes of its own call,
every row of the pair those of a call with that row alone, at K of two, three and four steps, of chunks of three, and longer
(members by themselves, the pair in two launches), on MLX arrays and tile-major."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,N2", [(5, 1152, 700, 33), (6, 2048, 2100, 512), (8, 2816, 520, 48), (7, 3968, 130, 1030), (8, 4096, 4096, 1024), (5, 8192, 96, 40), (8, 5376, 300, 64)])
def test_members_and_pair(ctx, M, K, N, N2):
    import aq_mi355
    say("rows in a grid", M, K, N, N2)
    xs = F.synthetic_x(M, K, seed=3200)
    x, raw = ctx.to_device(xs), [F.synthetic_affine(n, K, 4, 64, seed=3201 + i) for i, n in enumerate((N, N2, N))]
    mats = [DeviceAffine(ctx, *m) for m in raw]
    Ns, f32 = [N, N2, N], aq_mi355.AQ_OUT_F32
    tiled = [ctx.tile_weights(d.w, d.s, d.b, n, K) for d, n in zip(mats, Ns)] if K % 128 == 0 else None
    one, ys = ctx.alloc(M * max(Ns) * 4), [ctx.alloc(M * n * 4) for n in Ns]
    for flags, w, s, b in [(0, [d.w for d in mats], [d.s for d in mats], [d.b for d in mats])] + ([(aq_mi355.AQ_W_TILED, tiled, [None] * 3, [None] * 3)] if tiled else []):
        ctx.qmv_multi(x, w, s, b, ys, Ns, M, K, 64, 4, flags | f32)
        ctx.sync()
        assert ctx.last_variant(0).startswith("qmvd_multi_m8" if K <= 4096 else "qmvd_b4_m4_"), ctx.last_variant(0)
        for d, m, n, y in zip(mats, raw, Ns, ys):
            ctx.qmv(x, d.w, d.s, d.b, one, M, K, n, 64, 4, f32)
            ctx.sync()
            got = y.download(np.uint32, M * n)
            assert np.array_equal(got, one.download(np.uint32, M * n)), ("member", flags, n)
            check_accumulators(got.view(np.float32), F.reference_f64(xs, *m, 4, 64, K), "member of %d rows" % n)
        ctx.fill_zero(one)
        pair = [(w[0], s[0], b[0]), (w[2], s[2], b[2])]
        ctx.qmv_gate_up(x, *pair, one, M, K, N, 64, 4, aq_mi355.AQ_ACT_SILU, flags | f32)
        ctx.sync()
        assert ctx.last_variant(0) == "qmv_gate_up_diag", ctx.last_variant(0)
        got = one.download(np.uint32, M * N).reshape(M, N)
        for m in range(M):
            ctx.qmv_gate_up(x.ptr + m * K * 2, *pair, ys[0], 1, K, N, 64, 4, aq_mi355.AQ_ACT_SILU, flags | f32)
            ctx.sync()
            assert np.array_equal(ys[0].download(np.uint32, N), got[m]), ("pair", flags, m)
    for t in [x, one] + ys + mats + (tiled or []):
        t.free()
