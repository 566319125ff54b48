"""Shares of K added by the last workgroup of a tile: matrices and pairs at the edges of the tiles (rows and columns that are no whole
blocks of 32), two to many shares, beside matrices whose shares a second kernel adds (which of the members: tests/calls_on_host.cc); the
same bytes in every repetition, between other calls over the same workspace, from a call of the matrix alone and from replays of a graph."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, run_qmv, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,gs,M,K,Ns", [(4, 64, 65, 4096, (515, 130, 64)), (4, 32, 96, 3840, (1100, 33, 257)), (4, 128, 129, 8192, (1024, 512, 31)),
                                            (8, 64, 66, 3072, (3072, 96, 1000)), (8, 32, 200, 2048, (640, 513, 64)), (4, 64, 300, 2816, (704, 2050, 1)),
                                            (4, 32, 500, 8192, (2048, 72, 95)), (8, 64, 777, 10240, (2560, 256, 17)), (4, 64, 129, 2816, (3072, 96, 1000)),
                                            (4, 32, 300, 2048, (4096, 1024, 33)), (4, 128, 777, 2048, (1100, 33, 257)), (4, 64, 500, 4096, (3072, 96, 1000)),
                                            (4, 64, 777, 2048, (4096, 1024, 33)), (8, 64, 300, 4096, (2048, 513, 513)), (8, 32, 500, 2816, (3072, 96, 1000))])
def test_repeated(ctx, bits, gs, M, K, Ns):
    import aq_mi355
    say("share sums", bits, gs, M, K, Ns)
    x = F.synthetic_x(M, K, seed=3400)
    mats = [F.synthetic_affine(n, K, bits, gs, seed=3401 + i) for i, n in enumerate(Ns)]
    dws = [DeviceAffine(ctx, *m) for m in mats]
    alone = [run_qmv(ctx, x, d, M, K, n, gs, bits, True, fn="qmm").reshape(M, n) for d, n in zip(dws, Ns)]
    rows = sorted({0, 31, 32, M // 2, M - 1})
    for m, n, got in zip(mats, Ns, alone):
        check_accumulators(got[rows], F.reference_f64(x[rows], *m, bits, gs, K), "%d columns" % n)
    dx, f32 = ctx.to_device(x), aq_mi355.AQ_OUT_F32
    ys, gated = [ctx.alloc(M * n * 4) for n in Ns], ctx.alloc(M * Ns[0] * 4)
    pair = [(d.w, d.s, d.b) for d in (dws[0], dws[0])]

    def calls():
        ctx.qmm_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, bits, f32)
        ctx.qmv_gate_up(dx, *pair, gated, M, K, Ns[0], gs, bits, aq_mi355.AQ_ACT_SILU, f32)

    def results():
        ctx.sync()
        return [y.download(np.uint32, M * n) for y, n in zip(ys, Ns)] + [gated.download(np.uint32, M * Ns[0])]

    calls()
    first = results()
    for got, one in zip(first, alone):
        assert np.array_equal(got, one.view(np.uint32).reshape(-1))
    g = alone[0].astype(np.float64)
    assert np.allclose(first[-1].view(np.float32).reshape(M, -1), g * g / (1.0 + np.exp(np.clip(-g, -700, 700))), rtol=1e-5, atol=1e-6)
    ctx.capture_begin()
    calls()
    graph = ctx.capture_end()
    for _ in range(4):
        for y in ys + [gated]:
            ctx.fill_zero(y)
        ctx.graph_launch(graph)
        assert all(np.array_equal(a, b) for a, b in zip(results(), first))
        run_qmv(ctx, x[:40], dws[0], 40, K, Ns[0], gs, bits, True, fn="qmm")  # other contents for the workspace
        calls()
        assert all(np.array_equal(a, b) for a, b in zip(results(), first))
    ctx.graph_destroy(graph)
    for t in [dx, gated] + ys + dws:
        t.free()


def test_members_one_by_one():
    """A recorded call whose workspace holds a member at a time: the tickets of a later member are cleared by a launch of their own
    (tests/calls_on_host.cc looks at the launches), in every replay, whatever the workspace holds by then."""
    import aq_mi355
    M, K, Ns = 65, 2048, (515, 500, 130)
    say("share sums one by one")
    c = aq_mi355.Context(0)
    try:
        x = F.synthetic_x(M, K, seed=3500)
        mats = [F.synthetic_affine(n, K, 4, 64, seed=3501 + i) for i, n in enumerate(Ns)]
        dws = [DeviceAffine(c, *m) for m in mats]
        want = [run_qmv(c, x, d, M, K, n, 64, 4, True, fn="qmm") for d, n in zip(dws, Ns)]
        for m, got in zip(mats, want):
            check_accumulators(got, F.reference_f64(x, *m, 4, 64, K), "a member alone")
        dx, ys = c.to_device(x), [c.alloc(M * n * 4) for n in Ns]
        before = c.workspace_bytes()
        c.capture_begin()
        c.qmm_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, 64, 4, aq_mi355.AQ_OUT_F32)
        graph = c.capture_end()
        assert c.workspace_bytes() == before
        for _ in range(4):
            for y in ys:
                c.fill_zero(y)
            c.graph_launch(graph)
            c.sync()
            for y, n, one in zip(ys, Ns, want):
                assert np.array_equal(y.download(np.uint32, M * n), one.view(np.uint32).reshape(-1))
            run_qmv(c, x[::-1], dws[0], M, K, Ns[0], 64, 4, True, fn="qmm")  # other contents for the workspace
        c.graph_destroy(graph)
        for t in [dx] + ys + dws:
            t.free()
    finally:
        c.close()
