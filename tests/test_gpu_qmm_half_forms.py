"""The fp16-operand matmul kernels in groups of 32, with K shared out over workgroups, over several matrices in one grid and
as the gated pair.  Accumulators within the stated bounds of the float64 reference."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, run_qmv, say

pytestmark = pytest.mark.gpu

# edges of 32-, 64-, 128-, 192- and 256-row tiles; K of one block, a piece of a quad, shares of K of which the last is short
GROUP32 = [(5, 64, 40), (33, 192, 257), (64, 4032, 70), (65, 1088, 1001), (129, 704, 300), (509, 960, 2050), (200, 3840, 8200), (1030, 512, 4100)]


@pytest.mark.parametrize("M,K,N", GROUP32)
def test_groups_of_32(ctx, M, K, N):
    say("qmm group 32", M, K, N)
    words, s, b = F.synthetic_affine(N, K, 4, 32, seed=2400 + M)
    x = F.synthetic_x(M, K, seed=2401 + K)
    dw = DeviceAffine(ctx, words, s, b)
    acc = run_qmv(ctx, x, dw, M, K, N, 32, 4, True, fn="qmm")
    name = ctx.last_variant(1)
    assert name.startswith("qmmh_"), name
    cols = np.unique(np.r_[0, N - 1, np.random.default_rng(7).choice(N, min(N, 160), replace=False)])
    check_accumulators(acc[:, cols], F.reference_f64(x, words[cols], s[cols], b[cols], 4, 32, K), "%s M=%d K=%d N=%d" % (name, M, K, N))
    out = run_qmv(ctx, x, dw, M, K, N, 32, 4, False, fn="qmm")
    assert np.array_equal(out, F.f32_to_bf16_bits(acc).reshape(M, N))
    dw.free()


def test_groups_of_32_power_of_two_factors(ctx):
    """Rows of x and of the weights scaled by powers of two scale the fp32 results by exactly those powers."""
    M, K, N = 130, 512, 200
    say("qmm group 32 scaling", M, K, N)
    words, s, b = F.synthetic_affine(N, K, 4, 32, seed=2450)
    x = F.synthetic_x(M, K, seed=2451)
    rng = np.random.default_rng(3)
    row_pow, col_pow = rng.integers(-80, 60, M), rng.integers(-40, 40, N)
    scaled = lambda bits, p: F.f32_to_bf16_bits((F.bf16_bits_to_f32(bits) * np.exp2(p)[:, None]).astype(np.float32))
    dw, dw2 = DeviceAffine(ctx, words, s, b), DeviceAffine(ctx, words, scaled(s, col_pow), scaled(b, col_pow))
    base = run_qmv(ctx, x, dw, M, K, N, 32, 4, True, fn="qmm").reshape(M, N).astype(np.float64)
    rows = run_qmv(ctx, scaled(x, row_pow).reshape(x.shape), dw, M, K, N, 32, 4, True, fn="qmm").reshape(M, N)
    assert np.array_equal(rows, (base * np.exp2(row_pow)[:, None]).astype(np.float32))
    cols = run_qmv(ctx, x, dw2, M, K, N, 32, 4, True, fn="qmm").reshape(M, N)
    assert np.array_equal(cols, (base * np.exp2(col_pow)[None, :]).astype(np.float32))
    dw.free()
    dw2.free()


@pytest.mark.parametrize("gs,M,K,Ns", [(32, 70, 1024, (256, 64, 64)), (64, 300, 4096, (1024, 130, 256)), (128, 100, 2048, (512, 300)),
                                       (64, 40, 960, (600, 72)), (32, 20, 3840, (300, 41)), (64, 2048, 1024, (2048, 256, 256))])
def test_matrices_in_one_grid_have_the_bytes_of_their_own_calls(ctx, gs, M, K, Ns):
    """Members that share K out over workgroups beside members that do not; every one byte for byte its own aq_qmm call."""
    say("qmm multi", gs, M, K, Ns)
    mats = [F.synthetic_affine(n, K, 4, gs, seed=2500 + i) for i, n in enumerate(Ns)]
    x = F.synthetic_x(M, K, seed=2550)
    dws = [DeviceAffine(ctx, *m) for m in mats]
    alone = [run_qmv(ctx, x, d, M, K, n, gs, 4, True, fn="qmm") for d, n in zip(dws, Ns)]
    dx, ys = ctx.to_device(x), [ctx.alloc(M * n * 4) for n in Ns]
    import aq_mi355
    ctx.qmm_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, 4, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    for n, m, y, one in zip(Ns, mats, ys, alone):
        got = y.download(np.float32, M * n).reshape(M, n)
        assert np.array_equal(got.view(np.uint32), one.reshape(M, n).view(np.uint32))
        rows = sorted({0, M // 2, M - 1})
        check_accumulators(got[rows], F.reference_f64(x[rows], *m, 4, gs, K), "member of %d columns" % n)
    for t in [dx] + ys + dws:
        t.free()


@pytest.mark.parametrize("gs,M,K,N", [(32, 33, 960, 130), (32, 509, 1024, 515), (64, 65, 4096, 512), (64, 1030, 512, 2050), (128, 300, 2048, 264)])
def test_gated_pair(ctx, orc, gs, M, K, N):
    """act(gate . x) * (up . x) from the sums of the separate calls, whole or in shares of K."""
    import aq_mi355
    say("qmm gate|up", gs, M, K, N)
    gate, up = F.synthetic_affine(N, K, 4, gs, seed=2600), F.synthetic_affine(N, K, 4, gs, seed=2601)
    x = F.synthetic_x(M, K, seed=2602)
    dg, du = DeviceAffine(ctx, *gate), DeviceAffine(ctx, *up)
    g, u = (run_qmv(ctx, x, d, M, K, N, gs, 4, True, fn="qmm").reshape(M, N) for d in (dg, du))
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    for act in (aq_mi355.AQ_ACT_GELU_TANH, aq_mi355.AQ_ACT_SILU):
        ctx.qmv_gate_up(dx, (dg.w, dg.s, dg.b), (du.w, du.s, du.b), dy, M, K, N, gs, 4, act, aq_mi355.AQ_OUT_F32)
        ctx.sync()
        assert ctx.last_variant(0) == "qmv_gate_up_tiles"
        got = dy.download(np.float32, M * N).reshape(M, N)
        want = orc.act_multiply(act, g.reshape(-1), u.reshape(-1)).reshape(M, N)
        # the same fp32 sums; tanh and exp of the device library against the oracle's: a few fp32 ulp
        assert (np.abs(got - want) <= 4e-6 * np.abs(want) + 2.5e-7 * np.maximum(1.0, np.abs(g * u))).all()
        ctx.qmv_gate_up(dx, (dg.w, dg.s, dg.b), (du.w, du.s, du.b), dy, M, K, N, gs, 4, act, 0)
        ctx.sync()
        assert np.array_equal(dy.download(np.uint16, M * N), F.f32_to_bf16_bits(got).reshape(-1))
    for t in (dx, dy, dg, du):
        t.free()


def test_ragged_shares_of_k_few_rows(ctx):
    """5..32 rows of a narrow matrix whose K is no multiple of 256: the 32 x 256 tiles share K out too."""
    M, K, N = 12, 4032, 300
    say("few rows, ragged shares of K", M, K, N)
    words, s, b = F.synthetic_affine(N, K, 4, 64, seed=2700)
    x = F.synthetic_x(M, K, seed=2701)
    dw = DeviceAffine(ctx, words, s, b)
    acc = run_qmv(ctx, x, dw, M, K, N, 64, 4, True)
    assert ctx.last_variant(0).startswith("qmmt_"), ctx.last_variant(0)
    check_accumulators(acc, F.reference_f64(x, words, s, b, 4, 64, K), "ragged shares")
    dw.free()


@pytest.mark.parametrize("bits,gs,M,K,N", [(4, 64, 300, 4096, 4096), (4, 128, 130, 8192, 1024), (8, 64, 300, 4096, 4096), (4, 64, 40, 4032, 512),
                                           (4, 64, 97, 15360, 3840)])
def test_reserved_by_rows_and_columns_a_call_is_captured_on_its_kernels(bits, gs, M, K, N):
    """aq_reserve_workspace(M, K) holds all that a prefill call of that size needs, its partial tiles included: recorded into a
    graph it runs on the kernels of the eager call and gives its bytes; so does a call of fewer rows."""
    import aq_mi355
    say("qmm in a graph after reserving", bits, gs, M, K, N)
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=2720)
    x = F.synthetic_x(M, K, seed=2721)
    fresh = aq_mi355.Context(0)
    try:
        dw = DeviceAffine(fresh, words, s, b)
        dx, dy = fresh.to_device(x), fresh.alloc(M * N * 4)
        fresh.reserve_workspace(M, K)
        held = fresh.workspace_bytes()
        recorded = []
        for rows in (M, M - 3):
            fresh.capture_begin()
            fresh.qmm(dx, dw.w, dw.s, dw.b, dy, rows, K, N, gs, bits, aq_mi355.AQ_OUT_F32)
            recorded.append((rows, fresh.last_variant(1), fresh.capture_end()))
        for rows, name, graph in recorded:
            fresh.qmm(dx, dw.w, dw.s, dw.b, dy, rows, K, N, gs, bits, aq_mi355.AQ_OUT_F32)
            fresh.sync()
            want = dy.download(np.uint32, rows * N)
            assert name == fresh.last_variant(1) and name.startswith("qmmh"), (name, fresh.last_variant(1))
            assert fresh.workspace_bytes() == held
            for _ in range(3):
                fresh.fill_zero(dy)
                fresh.graph_launch(graph)
                fresh.sync()
                assert np.array_equal(dy.download(np.uint32, rows * N), want)
            fresh.graph_destroy(graph)
        for t in (dx, dy, dw):
            t.free()
    finally:
        fresh.close()


@pytest.mark.parametrize("bytes_too", [0, 1 << 20])
def test_several_matrices_captured_after_reserving(bytes_too):
    """aq_qmm_multi in a graph: with room for one matrix at a time (aq_reserve_workspace) or only for the copy of x and small
    shares of K, every member has the bytes of its own eager call or the call is refused, and nothing allocates."""
    import aq_mi355
    M, K, Ns = 200, 4096, (4096, 1024, 520)
    say("qmm multi in a graph", bytes_too)
    fresh = aq_mi355.Context(0)
    try:
        x = F.synthetic_x(M, K, seed=2730)
        dws = [DeviceAffine(fresh, *F.synthetic_affine(n, K, 4, 64, seed=2731 + i)) for i, n in enumerate(Ns)]
        dx, ys = fresh.to_device(x), [fresh.alloc(M * n * 4) for n in Ns]
        if bytes_too:
            fresh.reserve_workspace_bytes(M * K * 2 + bytes_too)
        else:
            fresh.reserve_workspace(M, K)
        held = fresh.workspace_bytes()
        call = lambda: fresh.qmm_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, 64, 4, aq_mi355.AQ_OUT_F32)
        fresh.capture_begin()
        refused = False
        try:
            call()
        except aq_mi355.AqError as e:
            assert bytes_too and e.code == aq_mi355.AQ_ERR_UNSUPPORTED
            refused = True
        graph = fresh.capture_end()
        assert fresh.workspace_bytes() == held and refused == bool(bytes_too)
        if not refused:
            for _ in range(3):
                for y in ys:
                    fresh.fill_zero(y)
                fresh.graph_launch(graph)
                fresh.sync()
                got = [y.download(np.uint32) for y in ys]
                for d, n, one in zip(dws, Ns, got):
                    assert np.array_equal(run_qmv(fresh, x, d, M, K, n, 64, 4, True, fn="qmm").view(np.uint32).reshape(-1), one)
        fresh.graph_destroy(graph)
        for t in [dx] + ys + dws:
            t.free()
    finally:
        fresh.close()
