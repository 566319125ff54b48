"""The gated pair and grids of several matrices on the tiles of 96 and 128 rows a wavefront and on the wide 8-bit ones, where the rule
picks them: K that ends inside a quad of blocks, whole and in shares of K, rows and columns that end inside a tile."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, run_qmv, say

pytestmark = pytest.mark.gpu

B4 = {"256x128": "qmmh_b4_mb4_nb2_wm2_wn2_s2c", "128x256": "qmmh_b4_mb4_nb2_wm1_wn4_s2c", "256x256": "qmmh_b4_mb4_nb2_wm2_wn4", "192x256": "qmmh_b4_mb3_nb2_wm2_wn4"}
B8 = {"128x128": "qmmh8_b8_mb2_nb2_wm2_wn2", "128x256": "qmmh8_b8_mb2_nb2_wm2_wn4", "64x256": "qmmh8_b8_mb2_nb2_wm1_wn4"}


def _operands(ctx, bits, gs, M, K, N, seed):
    m = F.synthetic_affine(N, K, bits, gs, seed=seed)
    return m, DeviceAffine(ctx, *m)


def _check_columns(acc, x, m, bits, gs, K, what):
    N = acc.shape[1]
    cols = np.unique(np.r_[0, N - 1, np.random.default_rng(5).choice(N, min(N, 60), replace=False)])
    check_accumulators(acc[:, cols], F.reference_f64(x, m[0][cols], m[1][cols], m[2][cols], bits, gs, K), what)


@pytest.mark.parametrize("bits,gs,M,K,N,tile", [(4, 32, 513, 1856, 3986, "256x128"), (4, 32, 200, 3904, 4758, "256x128"), (4, 32, 513, 3904, 5530, "128x256"),
                                                (4, 32, 200, 3904, 4179, "256x256"), (4, 32, 130, 3904, 2770, "192x256"), (4, 64, 513, 1856, 3986, "128x256"),
                                                (4, 64, 509, 1856, 4372, "256x128"), (4, 64, 130, 3904, 3675, "192x256"), (8, 32, 513, 3904, 6109, "128x256"),
                                                (8, 32, 130, 3904, 2147, "64x256"), (8, 32, 513, 832, 3986, "128x128"), (8, 64, 200, 3904, 4758, "128x256")])
def test_gated_pair(ctx, orc, bits, gs, M, K, N, tile):
    import aq_mi355
    say("gate|up on large tiles", bits, gs, M, K, N, tile)
    (gate, dg), (up, du) = (_operands(ctx, bits, gs, M, K, N, 5200 + i) for i in range(2))
    x = F.synthetic_x(M, K, seed=5202)
    g, u = (run_qmv(ctx, x, d, M, K, N, gs, bits, True, fn="qmm").reshape(M, N) for d in (dg, du))
    _check_columns(g, x, gate, bits, gs, K, tile)
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    act = aq_mi355.AQ_ACT_SILU
    ctx.qmv_gate_up(dx, (dg.w, dg.s, dg.b), (du.w, du.s, du.b), dy, M, K, N, gs, bits, act, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(1) == (B4 if bits == 4 else B8)[tile]
    got = dy.download(np.float32, M * N).reshape(M, N)
    want = orc.act_multiply(act, g.reshape(-1), u.reshape(-1)).reshape(M, N)
    # the same fp32 sums; exp of the device library against the oracle's: a few fp32 ulp
    assert (np.abs(got - want) <= 4e-6 * np.abs(want) + 2.5e-7 * np.maximum(1.0, np.abs(g * u))).all()
    for t in (dx, dy, dg, du):
        t.free()


@pytest.mark.parametrize("bits,gs,M,K,Ns", [(4, 32, 509, 3840, (4096, 2048, 2050)), (4, 64, 1030, 3904, (4096, 1024, 1001)), (8, 64, 777, 2560, (2048, 512, 515))])
def test_matrices_in_one_grid(ctx, bits, gs, M, K, Ns):
    """Members with long loops beside members in shares of K; every one byte for byte its own call."""
    import aq_mi355
    say("grid on large tiles", bits, gs, M, K, Ns)
    x = F.synthetic_x(M, K, seed=5300)
    mats, dws = zip(*(_operands(ctx, bits, gs, M, K, n, 5301 + i) for i, n in enumerate(Ns)))
    alone = [run_qmv(ctx, x, d, M, K, n, gs, bits, True, fn="qmm") for d, n in zip(dws, Ns)]
    dx, ys = ctx.to_device(x), [ctx.alloc(M * n * 4) for n in Ns]
    ctx.qmm_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, bits, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    for n, m, y, one in zip(Ns, mats, ys, alone):
        got = y.download(np.float32, M * n).reshape(M, n)
        assert np.array_equal(got.view(np.uint32), one.reshape(M, n).view(np.uint32))
        _check_columns(got, x, m, bits, gs, K, "member of %d columns" % n)
    for t in [dx] + ys + list(dws):
        t.free()
