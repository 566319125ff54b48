"""Two to four rows of x in groups of 32 and 128 where the dot2 kernels run one row: every row has the bytes of a call with that row alone, in
single calls, as members of a grid and in a gated pair; members that the block-MFMA shapes send to the token tiles beside them."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, say

pytestmark = pytest.mark.gpu


# (4 bit in groups of 128: 512 codes and whole sets of four rows of weights are the token tiles' shapes)
@pytest.mark.parametrize("bits,gs,M,K,Ns", [(4, 32, 2, 1216, (1537, 448, 33)), (4, 32, 2, 64, (16, 5)), (4, 32, 2, 4032, (1001, 2050)),
                                            (4, 128, 2, 1152, (1537, 384, 33)), (4, 128, 3, 896, (1000, 7)), (4, 128, 4, 1024, (1001, 256, 2)),
                                            (4, 128, 4, 14464, (203, 64)), (8, 128, 2, 128, (1, 64)), (8, 128, 3, 4096, (1030, 512, 33)),
                                            (8, 128, 4, 896, (1024, 256, 7)), (8, 128, 4, 7168, (300, 5))])
@pytest.mark.parametrize("f32", [True, False])
def test_rows_have_the_bytes_of_single_row_calls(ctx, bits, gs, M, K, Ns, f32):
    import aq_mi355
    say("bytes of rows", bits, gs, M, K, Ns, f32)
    flags, word, size = (aq_mi355.AQ_OUT_F32, np.uint32, 4) if f32 else (0, np.uint16, 2)
    xs = F.synthetic_x(M, K, seed=3600)
    x = ctx.to_device(xs)
    raw = [F.synthetic_affine(n, K, bits, gs, seed=3601 + i) for i, n in enumerate(Ns)]
    mats = [DeviceAffine(ctx, *m) for m in raw]
    one, ys = ctx.alloc(M * max(Ns) * size), [ctx.alloc(M * n * size) for n in Ns]
    ctx.qmv_multi(x, [d.w for d in mats], [d.s for d in mats], [d.b for d in mats], ys, list(Ns), M, K, gs, bits, flags)
    ctx.sync()
    for d, m, n, y in zip(mats, raw, Ns, ys):
        got = y.download(word, M * n).reshape(M, n)
        ctx.qmv(x, d.w, d.s, d.b, one, M, K, n, gs, bits, flags)
        ctx.sync()
        assert np.array_equal(got.reshape(-1), one.download(word, M * n)), ("member", n)
        if bits == 4 and gs == 128 and K % 512 == 0 and n % 4 == 0:
            assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
        else:
            assert ctx.last_variant(0).startswith("qmv_b%d_" % bits), ctx.last_variant(0)
            for r in range(M):
                ctx.qmv(x.ptr + r * K * 2, d.w, d.s, d.b, one, 1, K, n, gs, bits, flags)
                ctx.sync()
                assert np.array_equal(one.download(word, n), got[r]), (n, r)
        if f32:
            check_accumulators(got.view(np.float32), F.reference_f64(xs, *m, bits, gs, K), "member of %d rows" % n)
    N = Ns[0]
    pair = [(d.w, d.s, d.b) for d in (mats[0], DeviceAffine(ctx, *F.synthetic_affine(N, K, bits, gs, seed=3610)))]
    ctx.qmv_gate_up(x, *pair, one, M, K, N, gs, bits, aq_mi355.AQ_ACT_SILU, flags)
    ctx.sync()
    assert ctx.last_variant(0) == "qmv_gate_up_dot2", ctx.last_variant(0)
    got = one.download(word, M * N).reshape(M, N)
    for r in range(M):
        ctx.qmv_gate_up(x.ptr + r * K * 2, *pair, ys[0], 1, K, N, gs, bits, aq_mi355.AQ_ACT_SILU, flags)
        ctx.sync()
        assert np.array_equal(ys[0].download(word, N), got[r]), r
    for t in [x, one] + ys + mats + list(pair[1]):
        t.free()
