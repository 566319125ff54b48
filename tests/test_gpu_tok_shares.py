"""Token-tile calls that share K out over workgroups, that run 33..64 rows as two halves, and with eight sets of weight rows a
workgroup, at the edges of these choices.

Bounds: fp32 results within 2^-21 of the float64 product's 2-norm (eight roundings of 2^-24 on the way; partial tiles add one
per share, in order, of sums that are smaller than the result)."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, run_qmv, say

pytestmark = pytest.mark.gpu

# K of several passes (the last share or the last run shorter), rows of weights in fours or not; 33, 63 and 64 rows; the narrowest
# matrix of the halves; more than one round of eight sets
SHAPES = [(4, 64, 10, 14336, 77), (4, 64, 24, 16384, 529), (4, 64, 17, 9728, 2560), (4, 64, 32, 14400, 640), (4, 32, 21, 15360, 100),
          (4, 32, 16, 15296, 33), (4, 128, 32, 16256, 40), (8, 64, 9, 14336, 77), (8, 64, 32, 16320, 640), (8, 32, 20, 9792, 130),
          (8, 128, 7, 16384, 16)]
SHAPES += [(4, 64, 33, 1024, 529), (4, 64, 63, 2112, 1030), (4, 32, 64, 4096, 600), (4, 32, 33, 15360, 545), (4, 128, 47, 512, 4097),
           (8, 64, 64, 1024, 529), (8, 64, 33, 960, 2000), (8, 32, 63, 192, 1001), (8, 128, 40, 14336, 600)]
SHAPES += [(4, 64, 9, 256, 32770), (4, 32, 18, 64, 33000), (8, 64, 12, 64, 32800), (8, 128, 32, 128, 32769)]


@pytest.mark.parametrize("bits,gs,M,K,N", SHAPES)
def test_sums(ctx, bits, gs, M, K, N):
    say("token tile shares", bits, gs, M, K, N)
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=2400 + K)
    x = F.synthetic_x(M, K, seed=2401 + M)
    dw = DeviceAffine(ctx, words, s, b)
    acc = run_qmv(ctx, x, dw, M, K, N, gs, bits, True)
    assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
    ref = F.reference_f64(x, words, s, b, bits, gs, K)
    err = np.linalg.norm(acc.astype(np.float64).reshape(M, N) - ref) / np.linalg.norm(ref)
    print("error %.2e" % err)
    assert err <= 2.0 ** -21
    check_accumulators(acc, ref, "%d rows" % M)
    again = run_qmv(ctx, x, dw, M, K, N, gs, bits, True)
    assert np.array_equal(again.view(np.uint32), acc.view(np.uint32))
    out = run_qmv(ctx, x, dw, M, K, N, gs, bits, False)
    assert np.array_equal(out, F.f32_to_bf16_bits(acc).reshape(M, N))
    dw.free()


@pytest.mark.parametrize("bits,gs,M,K,Ns", [(4, 64, 12, 14336, (1000, 17, 4096)), (4, 64, 24, 8192, (2048, 530)), (4, 32, 21, 15360, (130, 64, 1)),
                                            (8, 64, 20, 9728, (512, 96)), (4, 64, 9, 5376, (4096, 2048, 2048)), (8, 64, 32, 5312, (2047, 4090, 2048)),
                                            (4, 32, 21, 6144, (1024, 6144, 1001)), (8, 32, 8, 5376, (4096, 2048, 2048)), (4, 128, 17, 8192, (8192, 1024)), (4, 64, 48, 4096, (1000, 530)), (8, 32, 33, 1024, (600, 700, 540))])
def test_members_have_the_bytes_of_their_own_calls(ctx, bits, gs, M, K, Ns):
    import aq_mi355
    say("token tile shares, members", bits, gs, M, K, Ns)
    x = F.synthetic_x(M, K, seed=2470)
    dws = [DeviceAffine(ctx, *F.synthetic_affine(n, K, bits, gs, seed=2471 + i)) for i, n in enumerate(Ns)]
    alone = [run_qmv(ctx, x, d, M, K, n, gs, bits, True) for d, n in zip(dws, Ns)]
    dx, ys = ctx.to_device(x), [ctx.alloc(M * n * 4) for n in Ns]
    ctx.qmv_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, bits, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
    for n, y, one in zip(Ns, ys, alone):
        assert np.array_equal(y.download(np.uint32, M * n), one.view(np.uint32).reshape(-1)), "member of %d rows" % n
    for t in [dx] + ys + dws:
        t.free()


@pytest.mark.parametrize("bits,gs,M,K,N", [(4, 64, 12, 14336, 77), (4, 32, 21, 15360, 100), (8, 64, 32, 9728, 1030), (4, 64, 33, 1024, 1000),
                                           (4, 128, 64, 256, 16384), (8, 64, 48, 2048, 529)])
def test_gated_pair(ctx, orc, bits, gs, M, K, N):
    import aq_mi355
    say("token tile shares, gate|up", bits, gs, M, K, N)
    mats = [F.synthetic_affine(N, K, bits, gs, seed=2480 + i) for i in range(2)]
    x = F.synthetic_x(M, K, seed=2482)
    g, u = (F.reference_f64(x, *m, bits, gs, K) for m in mats)
    dws = [DeviceAffine(ctx, *m) for m in mats]
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    ctx.qmv_gate_up(dx, *((d.w, d.s, d.b) for d in dws), dy, M, K, N, gs, bits, aq_mi355.AQ_ACT_SILU, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0) == "qmv_gate_up_tok"
    got, want = dy.download(np.float32, M * N).reshape(M, N), g / (1.0 + np.exp(np.minimum(-g, 700.0))) * u
    # every sum within 2^-21 of the rms of its matrix's, the slope of silu up to 1.1, tanh and exp a few fp32 ulp
    tol = 8 * 2.0 ** -21 * (1.1 * np.abs(u) * np.sqrt(np.mean(g * g)) + np.abs(g) * np.sqrt(np.mean(u * u))) + 4e-6 * np.abs(want) + 1e-30
    assert (np.abs(got - want) <= tol).all()
    for t in [dx, dy] + dws:
        t.free()


@pytest.mark.parametrize("bits,gs,K,N", [(4, 64, 8192, 4096), (4, 64, 4736, 1985), (8, 64, 14336, 700), (4, 32, 15360, 545)])
def test_a_row_has_the_same_bytes_in_calls_of_9_to_32_rows(bits, gs, K, N):
    """... and of 33 to 64; eager, and recorded on a context that has never run anything."""
    import aq_mi355
    say("token tiles, rows across row counts", bits, gs, K, N)
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=2490)
    x = F.synthetic_x(64, K, seed=2491)
    fresh = aq_mi355.Context(0)
    try:
        dw, dx, dy = DeviceAffine(fresh, words, s, b), fresh.to_device(x), fresh.alloc(64 * N * 4)
        call = lambda m: fresh.qmv(dx, dw.w, dw.s, dw.b, dy, m, K, N, gs, bits, aq_mi355.AQ_OUT_F32)
        held = fresh.workspace_bytes()
        for counts in ((9, 12, 16, 17, 24, 28, 32), (33, 48, 64)):
            want = None
            for m in counts:
                fresh.capture_begin()
                call(m)
                graph = fresh.capture_end()
                assert fresh.last_variant(0).startswith("qmvt_"), fresh.last_variant(0)
                for replay in range(3):
                    fresh.fill_zero(dy)
                    fresh.graph_launch(graph)
                    fresh.sync()
                    got = dy.download(np.uint32, m * N).reshape(m, N)
                    want = got if want is None else want
                    assert np.array_equal(got[:len(want)], want[:m]), (m, replay)
                    call(m)
                    fresh.sync()
                    assert np.array_equal(dy.download(np.uint32, m * N).reshape(m, N), got), (m, replay)
                want = got
                fresh.graph_destroy(graph)
        assert fresh.workspace_bytes() == held
        check_accumulators(want.view(np.float32), F.reference_f64(x, words, s, b, bits, gs, K), "64 rows")
        for t in (dw, dx, dy):
            t.free()
    finally:
        fresh.close()


def test_capture_without_a_workspace():
    """A call that shares K out is captured on a context that has never run anything, and again after eager calls."""
    import aq_mi355
    M, K, N = 24, 14336, 700
    say("token tile shares in a graph", M, K, N)
    words, s, b = F.synthetic_affine(N, K, 4, 64, seed=2490)
    x = F.synthetic_x(M, K, seed=2491)
    ref = F.reference_f64(x, words, s, b, 4, 64, K)
    fresh = aq_mi355.Context(0)
    try:
        dw = DeviceAffine(fresh, words, s, b)
        dx, dy = fresh.to_device(x), fresh.alloc(M * N * 4)
        call = lambda: fresh.qmv(dx, dw.w, dw.s, dw.b, dy, M, K, N, 64, 4, aq_mi355.AQ_OUT_F32)
        for _ in range(2):
            fresh.capture_begin()
            call()
            graph = fresh.capture_end()
            for _ in range(3):
                fresh.fill_zero(dy)
                fresh.graph_launch(graph)
                fresh.sync()
                check_accumulators(dy.download(np.float32, M * N).copy(), ref, "replay")
            fresh.graph_destroy(graph)
            call()
            fresh.sync()
            check_accumulators(dy.download(np.float32, M * N).copy(), ref, "eager")
        for t in (dw, dx, dy):
            t.free()
    finally:
        fresh.close()


@pytest.mark.parametrize("reserve", [0, 1 << 20])
def test_members_apart_move_the_workspace(reserve):
    """A member that runs by itself, ahead of the grid, needs more workspace than the grid's partial tiles."""
    import aq_mi355
    M, K, Ns, gs, bits = 40, 14336, (600, 500, 1000), 64, 4
    say("token tile shares, members apart", reserve)
    x = F.synthetic_x(M, K, seed=2495)
    mats = [F.synthetic_affine(n, K, bits, gs, seed=2496 + i) for i, n in enumerate(Ns)]
    fresh = aq_mi355.Context(0)
    try:
        if reserve:
            fresh.reserve_workspace_bytes(reserve)
        dws = [DeviceAffine(fresh, *m) for m in mats]
        dx, ys = fresh.to_device(x), [fresh.alloc(M * n * 4) for n in Ns]
        fresh.qmv_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, bits, aq_mi355.AQ_OUT_F32)
        fresh.sync()
        for n, d, y in zip(Ns, dws, ys):
            alone = run_qmv(fresh, x, d, M, K, n, gs, bits, True)
            assert np.array_equal(y.download(np.uint32, M * n), alone.view(np.uint32).reshape(-1)), "member of %d rows" % n
        for t in [dx] + ys + dws:
            t.free()
    finally:
        fresh.close()
