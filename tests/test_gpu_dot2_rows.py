"""Two to eight rows of x at a K that the diagonal-MFMA kernels do not take (4 bit: up to 1024, no multiple of 128, beyond 16384; 8 bit: two to
four rows of small matrices, alone or beside one that the token-tile kernels run): several matrices
in one grid and a gated pair in one launch per four rows, every member with the bytes of its own call, every row of the pair with those of a
call with that row alone."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,M,K,Ns", [(4, 2, 64, (1, 33)), (4, 3, 1024, (700, 130, 7)), (4, 4, 832, (1088, 320, 320)), (4, 5, 1216, (1536, 448, 448)), (4, 7, 3008, (130, 1030)),
                                    (4, 8, 960, (1001, 64, 17, 2)), (4, 6, 16448, (96, 40)), (8, 2, 64, (1, 33)), (8, 3, 832, (1088, 320, 320)), (8, 4, 896, (1030, 256, 256)), (8, 4, 1216, (700, 7, 5000)), (8, 2, 3008, (96, 3072, 130))])
@pytest.mark.parametrize("f32", [True, False])
def test_members_and_pair(ctx, bits, M, K, Ns, f32):
    import aq_mi355
    say("dot2 rows", bits, M, K, Ns, f32)
    xs = F.synthetic_x(M, K, seed=3500)
    x = ctx.to_device(xs)
    raw = [F.synthetic_affine(n, K, bits, 64, seed=3501 + i) for i, n in enumerate(Ns)]
    mats = [DeviceAffine(ctx, *m) for m in raw]
    flags, word, size = (aq_mi355.AQ_OUT_F32, np.uint32, 4) if f32 else (0, np.uint16, 2)
    one, ys = ctx.alloc(M * max(Ns) * size), [ctx.alloc(M * n * size) for n in Ns]
    ctx.qmv_multi(x, [d.w for d in mats], [d.s for d in mats], [d.b for d in mats], ys, list(Ns), M, K, 64, bits, flags)
    ctx.sync()
    small = all(bits == 4 or n * K < 4 << 20 for n in Ns)
    assert ctx.last_variant(0).startswith(("qmvr_multi_dot2" if bits == 4 else "qmvr8_multi_dot2") if small else "qmvt_"), ctx.last_variant(0)
    for d, m, n, y in zip(mats, raw, Ns, ys):
        ctx.qmv(x, d.w, d.s, d.b, one, M, K, n, 64, bits, flags)
        ctx.sync()
        got = y.download(word, M * n)
        assert np.array_equal(got, one.download(word, M * n)), n
        if f32:
            check_accumulators(got.view(np.float32).reshape(M, n), F.reference_f64(xs, *m, bits, 64, K), "member of %d rows" % n)
    gate, N = mats[0], Ns[0]
    up = DeviceAffine(ctx, *F.synthetic_affine(N, K, bits, 64, seed=3510))
    pair = [(gate.w, gate.s, gate.b), (up.w, up.s, up.b)]
    ctx.qmv_gate_up(x, *pair, one, M, K, N, 64, bits, aq_mi355.AQ_ACT_SILU, flags)
    ctx.sync()
    assert ctx.last_variant(0) == "qmv_gate_up_dot2", ctx.last_variant(0)
    got = one.download(word, M * N).reshape(M, N)
    for m in range(M):
        ctx.qmv_gate_up(x.ptr + m * K * 2, *pair, ys[0], 1, K, N, 64, bits, aq_mi355.AQ_ACT_SILU, flags)
        ctx.sync()
        assert np.array_equal(ys[0].download(word, N), got[m]), m
    for t in [x, one, up] + ys + mats:
        t.free()
