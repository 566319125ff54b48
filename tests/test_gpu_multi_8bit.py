"""Several 8-bit matrices in one grid: every member has the bytes of its own call, on the diagonal kernels (K of 2048, 4096, 8192 up
to 40 Mi codes), on the dot2 kernel (other K, other groups, one row), or apart where the members' own calls differ."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,gs,Ns,K", [(1, 64, (64, 200), 4096), (1, 64, (4096, 1024, 1030), 4096), (2, 64, (96, 160), 2048), (4, 64, (50, 301), 4096),
                                       (3, 64, (33, 17, 1, 90), 8192), (1, 64, (10300, 40), 4096), (1, 32, (64, 200, 7), 2560), (1, 128, (300, 21), 1536),
                                       (1, 64, (16500, 50), 2560), (1, 64, (1, 3000), 192), (2, 32, (70, 40), 4096), (4, 64, (64, 65), 2048)])
@pytest.mark.parametrize("offset", [0, 2])
def test_members_have_the_bytes_of_their_own_calls(ctx, M, gs, Ns, K, offset):
    import aq_mi355
    say("8 bit multi", M, gs, Ns, K, offset)
    x = ctx.to_device(F.synthetic_x(M, K, seed=2900))
    mats, held = [], []
    for i, n in enumerate(Ns):
        words, s, b = F.synthetic_affine(n, K, 8, gs, seed=2901 + i)
        # the last member's scales at an offset that the diagonal kernels do not take
        off = offset if i == len(Ns) - 1 else 0
        sb = [ctx.to_device(np.concatenate([np.zeros(off // 2, np.uint16), np.ravel(t)])) for t in (s, b)]
        held += [ctx.to_device(words)] + sb
        mats.append((held[-3].ptr, sb[0].ptr + off, sb[1].ptr + off))
    one, ys = ctx.alloc(M * max(Ns) * 4), [ctx.alloc(M * n * 4) for n in Ns]
    ctx.qmv_multi(x, [m[0] for m in mats], [m[1] for m in mats], [m[2] for m in mats], ys, list(Ns), M, K, gs, 8, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    diag = [gs == 64 and n * K <= 40 << 20 and (K in (4096, 8192) or (K == 2048 and M <= 2)) for n in Ns]
    name = ctx.last_variant(0)
    if all(diag) and offset == 0:
        assert name == "qmv8_multi_diag", name
    elif M == 1 and not any(diag):
        assert name == "qmv8_multi_dot2", name
    else:  # in the token tiles' grid, or apart
        assert not name.startswith("qmv8_multi"), name
    for n, m, y in zip(Ns, mats, ys):
        ctx.qmv(x, m[0], m[1], m[2], one, M, K, n, gs, 8, aq_mi355.AQ_OUT_F32)
        ctx.sync()
        assert np.array_equal(y.download(np.uint32, M * n), one.download(np.uint32, M * n)), "member of %d rows" % n
    for t in held + ys + [x, one]:
        t.free()
