"""Gathered projections of many routes, grouped by expert on the device: against the per-route kernels' contract (the
float64 reference per route), with ids and rows of x out of range, experts without a route and experts with more routes than
a tile has rows."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, say

pytestmark = pytest.mark.gpu


def _ids(rng, routes, E, skew):
    """Expert of each route: at random, or most of them one expert with some experts left out."""
    if not skew:
        return rng.integers(0, E, routes).astype(np.int32)
    ids = rng.integers(0, max(1, E // 2), routes)
    ids[rng.random(routes) < 0.6] = E - 1
    return ids.astype(np.int32)


# tiles of 32, 64, 128 and 256 rows, token tiles of 16 and 32; K and N that end inside a tile; every width and group size
CASES = [(4, 64, 300, 8, 704, 130, False), (4, 64, 300, 8, 704, 130, True), (4, 32, 700, 6, 512, 264, True), (4, 128, 90, 3, 256, 40, False),
         (4, 64, 70, 16, 2816, 72, False), (4, 32, 65, 40, 2048, 64, True), (8, 64, 200, 32, 1088, 96, True), (8, 32, 700, 8, 320, 33, False),
         (4, 64, 1000, 2, 192, 515, True)]


@pytest.mark.parametrize("bits,gs,routes,E,K,N,skew", CASES)
def test_grouped_gather(ctx, orc, bits, gs, routes, E, K, N, skew):
    import aq_mi355
    say("grouped gather", bits, gs, routes, E, K, N, skew)
    rng = np.random.default_rng(routes + K)
    expert_rows, gate_base, up_base = 2 * ((N + 15) // 16 * 16), 0, (N + 15) // 16 * 16
    words, s, b = F.synthetic_affine(E * expert_rows, K, bits, gs, seed=2800 + K)
    x_rows = routes // 2
    x = F.synthetic_x(x_rows, K, seed=2801)
    rhs, lhs = _ids(rng, routes, E, skew), rng.integers(0, x_rows, routes).astype(np.int32)
    bad = {3: "rhs", 11: "rhs", 20: "lhs", routes - 1: "lhs"}
    rhs[3], rhs[11], lhs[20], lhs[routes - 1] = -1, E, x_rows, -5
    dw = DeviceAffine(ctx, words, s, b)
    dx, dl, dr, dy = ctx.to_device(x), ctx.to_device(lhs), ctx.to_device(rhs), ctx.alloc(routes * N * 4)
    refs = {}
    for base in (gate_base, up_base):
        ctx.fill_zero(dy)
        ctx.gather_qmv(dx, dw.w, dw.s, dw.b, dl, dr, dy, routes, x_rows, K, N, E, expert_rows, base, gs, bits, aq_mi355.AQ_OUT_F32)
        ctx.sync()
        assert "grouped" in ctx.last_variant(0), ctx.last_variant(0)
        got = dy.download(np.float32, routes * N).reshape(routes, N)
        ref = np.zeros((routes, N))
        for e in range(E):
            z = [r for r in np.nonzero(rhs == e)[0] if r not in bad]
            if z:
                rows = slice(e * expert_rows + base, e * expert_rows + base + N)
                ref[z] = F.reference_f64(x[lhs[z]], words[rows], s[rows], b[rows], bits, gs, K)
        assert not got[list(bad)].any(), "ids out of range give zeros"
        check_accumulators(got, ref, "grouped gather, rows from %d" % base)
        refs[base] = got
        out = ctx.alloc(routes * N * 2)
        ctx.gather_qmv(dx, dw.w, dw.s, dw.b, dl, dr, out, routes, x_rows, K, N, E, expert_rows, base, gs, bits)
        ctx.sync()
        assert np.array_equal(out.download(np.uint16, routes * N), F.f32_to_bf16_bits(got).reshape(-1))
        out.free()
    ctx.fill_zero(dy)
    ctx.gather_qmv_gate_up(dx, dw.w, dw.s, dw.b, dl, dr, dy, routes, x_rows, K, N, E, expert_rows, gate_base, up_base, gs, bits,
                           aq_mi355.AQ_ACT_SILU, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert "grouped" in ctx.last_variant(0), ctx.last_variant(0)
    got = dy.download(np.float32, routes * N).reshape(routes, N)
    g, u = refs[gate_base], refs[up_base]
    want = orc.act_multiply(aq_mi355.AQ_ACT_SILU, g.reshape(-1), u.reshape(-1)).reshape(routes, N)
    # the same fp32 sums; exp of the device library against the oracle's: a few fp32 ulp
    assert (np.abs(got - want) <= 4e-6 * np.abs(want) + 2.5e-7 * np.maximum(1.0, np.abs(g * u))).all()
    for t in (dx, dl, dr, dy, dw):
        t.free()


def test_grouped_gather_captured(ctx):
    """Recorded into a graph and replayed over changing ids: every replay equals the eager call."""
    import aq_mi355
    routes, E, K, N = 130, 4, 512, 64
    say("grouped gather in a graph")
    rng = np.random.default_rng(5)
    words, s, b = F.synthetic_affine(E * N, K, 4, 64, seed=2900)
    x = F.synthetic_x(routes, K, seed=2901)
    dw = DeviceAffine(ctx, words, s, b)
    dx, dl, dr, dy = ctx.to_device(x), ctx.to_device(np.arange(routes, dtype=np.int32)), ctx.alloc(routes * 4), ctx.alloc(routes * N * 4)
    call = lambda: ctx.gather_qmv(dx, dw.w, dw.s, dw.b, dl, dr, dy, routes, routes, K, N, E, N, 0, 64, 4, aq_mi355.AQ_OUT_F32)
    eager, sets = [], [rng.integers(0, E, routes).astype(np.int32) for _ in range(3)]
    for ids in sets:
        dr.upload(ids)
        call()
        ctx.sync()
        eager.append(dy.download(np.float32, routes * N).copy())
    ctx.capture_begin()
    call()
    graph = ctx.capture_end()
    for ids, want in zip(sets, eager):
        ctx.fill_zero(dy)
        dr.upload(ids)
        ctx.graph_launch(graph)
        ctx.sync()
        assert np.array_equal(dy.download(np.uint32, routes * N), want.view(np.uint32))
    ctx.graph_destroy(graph)
    for t in (dx, dl, dr, dy, dw):
        t.free()


def test_two_streams_share_one_workspace(ctx):
    """Grouped gathers keep their lists in the context's workspace: calls that alternate between two streams give what they
    give on one."""
    import ctypes
    say("grouped gathers on two streams")
    hip = ctypes.CDLL("libamdhip64.so")
    streams = [ctypes.c_void_p() for _ in range(2)]
    for st in streams:
        assert hip.hipStreamCreateWithFlags(ctypes.byref(st), 1) == 0
    jobs = []
    for i, (routes, E, K, N) in enumerate([(2000, 4, 1024, 512), (300, 16, 512, 256)]):
        rng = np.random.default_rng(60 + i)
        dw = DeviceAffine(ctx, *F.synthetic_affine(E * N, K, 4, 64, seed=2950 + i))
        held = [ctx.to_device(F.synthetic_x(routes, K, seed=2960 + i)), ctx.to_device(np.arange(routes, dtype=np.int32)),
                ctx.to_device(rng.integers(0, E, routes).astype(np.int32)), ctx.alloc(routes * N * 2)]
        dx, dl, dr, dy = held
        call = lambda a=(dx, dw.w, dw.s, dw.b, dl, dr, dy, routes, routes, K, N, E, N, 0, 64, 4): ctx.gather_qmv(*a)
        call()
        ctx.sync()
        jobs.append((call, dy, dy.download(np.uint16).copy(), held + [dw]))
    try:
        for _ in range(10):
            for _, dy, _, _ in jobs:
                ctx.fill_zero(dy)
            ctx.sync()
            for _ in range(3):
                for st, (call, _, _, _) in zip(streams, jobs):
                    assert ctx.lib.aq_use_stream(ctx.handle, st) == 0
                    call()
            for st, (_, dy, want, _) in zip(streams, jobs):
                assert hip.hipStreamSynchronize(st) == 0
            assert ctx.lib.aq_use_own_stream(ctx.handle) == 0
            for _, dy, want, _ in jobs:
                assert np.array_equal(dy.download(np.uint16), want)
    finally:
        ctx.lib.aq_use_own_stream(ctx.handle)
    for st in streams:
        hip.hipStreamDestroy(st)
    for _, _, _, held in jobs:
        for t in held:
            t.free()


def test_stream_destroyed_before_the_context_leaves_it(ctx):
    import ctypes
    say("stream destroyed before it is left")
    hip = ctypes.CDLL("libamdhip64.so")
    M, K, N = 40, 512, 64
    dw = DeviceAffine(ctx, *F.synthetic_affine(N, K, 4, 32, seed=2990))
    dx, dy = ctx.to_device(F.synthetic_x(M, K, seed=2991)), ctx.alloc(M * N * 2)
    call = lambda: ctx.qmm(dx, dw.w, dw.s, dw.b, dy, M, K, N, 32, 4)
    call()
    ctx.sync()
    want = dy.download(np.uint16).copy()
    for _ in range(3):
        ctx.fill_zero(dy)
        ctx.sync()
        st = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(st), 1) == 0
        assert ctx.lib.aq_use_stream(ctx.handle, st) == 0
        call()
        assert hip.hipStreamSynchronize(st) == 0 and hip.hipStreamDestroy(st) == 0
        assert ctx.lib.aq_use_own_stream(ctx.handle) == 0
        assert np.array_equal(dy.download(np.uint16), want)
        call()
        ctx.sync()
        assert np.array_equal(dy.download(np.uint16), want)
    for t in (dx, dy, dw):
        t.free()


def test_recorded_calls_outlive_a_larger_workspace(orc):
    """A gather of many routes and matmuls in groups of 32, recorded over the workspace, are replayed after it has moved (other
    calls asked for more); recorded where it has no room they run on the kernels that need none."""
    import aq_mi355
    say("recorded calls, workspace moved")
    fresh = aq_mi355.Context(0)
    try:
        routes, E, K, N, M = 300, 4, 512, 64, 40
        rng = np.random.default_rng(6)
        x = F.synthetic_x(routes, K, seed=2970)
        rhs = rng.integers(0, E, routes).astype(np.int32)
        mats = [F.synthetic_affine(E * N, K, 4, 64, seed=2971), F.synthetic_affine(N, K, 4, 32, seed=2972), F.synthetic_affine(2 * N, K, 4, 32, seed=2973)]
        dws = [DeviceAffine(fresh, *m) for m in mats]
        dx, dl, dr = fresh.to_device(x), fresh.to_device(np.arange(routes, dtype=np.int32)), fresh.to_device(rhs)
        ys = [fresh.alloc(routes * N * 4), fresh.alloc(M * N * 4), fresh.alloc(M * 2 * N * 4)]
        gather64 = np.zeros((routes, N))
        for e in range(E):
            rows = slice(e * N, (e + 1) * N)
            gather64[rhs == e] = F.reference_f64(x[rhs == e], mats[0][0][rows], mats[0][1][rows], mats[0][2][rows], 4, 64, K)
        want = [gather64] + [F.reference_f64(x[:M], *m, 4, 32, K) for m in mats[1:]]

        def step():
            d = dws[0]
            fresh.gather_qmv(dx, d.w, d.s, d.b, dl, dr, ys[0], routes, routes, K, N, E, N, 0, 64, 4, aq_mi355.AQ_OUT_F32)
            names = [fresh.last_variant(0)]
            fresh.qmm_multi(dx, [d.w for d in dws[1:]], [d.s for d in dws[1:]], [d.b for d in dws[1:]], ys[1:], [N, 2 * N], M, K, 32, 4,
                            aq_mi355.AQ_OUT_F32)
            return names + [fresh.last_variant(1)]

        def record():
            fresh.capture_begin()
            names = step()
            return fresh.capture_end(), names

        def replay(graph, what):
            for i in range(3):
                for y in ys:
                    fresh.fill_zero(y)
                fresh.graph_launch(graph)
                fresh.sync()
                for y, ref in zip(ys, want):
                    check_accumulators(y.download(np.float32, ref.size), ref, "%s, replay %d" % (what, i))

        bare, names = record()  # a context that has run nothing: no workspace
        assert "grouped" not in names[0] and names[1] == "qmv_generic", names
        step()
        fresh.sync()
        over, names = record()
        assert "grouped" in names[0] and names[1].startswith("qmmh_"), names
        replay(over, "before")
        fresh.reserve_workspace_bytes(64 << 20)
        fresh.gather_qmv(dx, dws[0].w, dws[0].s, dws[0].b, dl, dr, ys[0], routes, routes, K, N, E, N, 0, 64, 4, aq_mi355.AQ_OUT_F32)
        replay(over, "after")
        replay(bare, "without scratch")
        for g in (over, bare):
            fresh.graph_destroy(g)
        for t in [dx, dl, dr] + ys + dws:
            t.free()
    finally:
        fresh.close()


@pytest.mark.parametrize("offset", [0, 2])
def test_gather_act_of_many_routes(ctx, orc, offset):
    """bf16(act(gate) * up) gathered: where the activations are not 16-byte aligned the product lies in the workspace, and the
    gather behind it leaves that alone."""
    import aq_mi355
    routes, E, K, N = 200, 4, 512, 72
    say("gather of formed activations", offset)
    rng = np.random.default_rng(8)
    words, s, b = F.synthetic_affine(E * N, K, 4, 64, seed=2980)
    gate, up = F.synthetic_x(routes, K, seed=2981), F.synthetic_x(routes, K, seed=2982)
    rhs, lhs = rng.integers(0, E, routes).astype(np.int32), rng.permutation(routes).astype(np.int32)
    pad = lambda a: np.concatenate([np.zeros(offset // 2, np.uint16), a.reshape(-1)])
    dw = DeviceAffine(ctx, words, s, b)
    dg, du, dl, dr, dy = (ctx.to_device(pad(gate)), ctx.to_device(pad(up)), ctx.to_device(lhs), ctx.to_device(rhs), ctx.alloc(routes * N * 4))
    product = ctx.alloc(routes * K * 2)
    ctx.act_mul(dg.ptr + offset, du.ptr + offset, product, routes * K, aq_mi355.AQ_ACT_SILU)
    ctx.sync()
    x = product.download(np.uint16, routes * K).reshape(routes, K)
    ref = np.zeros((routes, N))
    for e in range(E):
        z, rows = np.nonzero(rhs == e)[0], slice(e * N, (e + 1) * N)
        ref[z] = F.reference_f64(x[lhs[z]], words[rows], s[rows], b[rows], 4, 64, K)
    for _ in range(2):
        ctx.fill_zero(dy)
        ctx.gather_qmv_act(dg.ptr + offset, du.ptr + offset, dw.w, dw.s, dw.b, dl, dr, dy, routes, routes, K, N, E, N, 0, 64, 4,
                           aq_mi355.AQ_ACT_SILU, aq_mi355.AQ_OUT_F32)
        ctx.sync()
        check_accumulators(dy.download(np.float32, routes * N), ref, "gather of formed activations")
    for t in (dg, du, dl, dr, dy, product, dw):
        t.free()
