"""Routes grouped by expert on tiles in blocks of 16 routes: K that ends in a half step, a step, inside a segment of scales and behind
one, columns that end inside a strip, experts of no route, of fewer than 16, 32, 48 and of several chunks; rows of x read by
several routes, by one, and all the first."""
import numpy as np
import pytest

import fixtures as F
import test_gpu_moe_grouped as grouped
from gpu_util import DeviceAffine, check_accumulators, say

pytestmark = pytest.mark.gpu


# routes, experts, K, N (1.4 tiles a CU of 256 columns and more)
@pytest.mark.parametrize("gs,routes,E,K,N,skew", [(64, 260, 80, 256, 1030, False), (64, 1900, 80, 320, 1033, False), (64, 700, 128, 704, 776, True),
                                                  (64, 2600, 80, 1088, 1030, True), (32, 1900, 80, 128, 1030, False), (32, 1200, 100, 576, 1028, True),
                                                  (128, 1900, 80, 640, 1030, False), (128, 1500, 100, 2176, 1024, False),
                                                  # the longest list beside the pass over x, and one in a launch of its own (tests/calls_on_host.cc)
                                                  (64, 5056, 128, 256, 776, False), (64, 5057, 128, 256, 776, True)])
def test_blocks(ctx, orc, gs, routes, E, K, N, skew):
    grouped.test_grouped_gather(ctx, orc, 4, gs, routes, E, K, N, skew)
    assert ctx.last_variant(0) == "gather_gate_up_grouped_blocks", ctx.last_variant(0)


@pytest.mark.parametrize("x_rows,use_lhs", [(7, True), (900, True), (5, False)])
def test_rows_of_x(ctx, x_rows, use_lhs):
    import aq_mi355
    routes, E, K, N = 800, 96, 448, 1024
    say("blocks of routes, rows of x", x_rows, use_lhs)
    rng = np.random.default_rng(x_rows)
    words, s, b = F.synthetic_affine(E * N, K, 4, 64, seed=3100)
    x = F.synthetic_x(x_rows, K, seed=3101)
    x[x_rows // 2, 5] = 0x7F80  # an infinity stays in its row
    rhs, lhs = rng.integers(0, E, routes).astype(np.int32), rng.integers(0, x_rows, routes).astype(np.int32)
    if not use_lhs:
        lhs[:] = 0
    dw = DeviceAffine(ctx, words, s, b)
    dx, dl, dr, dy = ctx.to_device(x), ctx.to_device(lhs), ctx.to_device(rhs), ctx.alloc(routes * N * 4)
    ctx.gather_qmv(dx, dw.w, dw.s, dw.b, dl if use_lhs else None, dr, dy, routes, x_rows, K, N, E, N, 0, 64, 4, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0) == "gather_grouped_blocks", ctx.last_variant(0)
    got = dy.download(np.float32, routes * N).reshape(routes, N)
    plain = lhs != x_rows // 2
    assert not use_lhs or not np.isfinite(got[~plain]).any()
    ref = np.zeros((routes, N))
    for e in range(E):
        z, rows = np.nonzero((rhs == e) & plain)[0], slice(e * N, (e + 1) * N)
        if len(z):
            ref[z] = F.reference_f64(x[lhs[z]], words[rows], s[rows], b[rows], 4, 64, K)
    check_accumulators(got[plain], ref[plain], "blocks of routes")
    for t in (dx, dl, dr, dy, dw):
        t.free()


@pytest.mark.parametrize("gs,K", [(64, 704), (32, 576), (128, 1280)])
def test_no_further_from_float64_than_tiles_of_32_routes(ctx, gs, K):
    """The first experts' routes once among those of many experts (blocks of 16) and once by themselves, too few workgroups for blocks: the
    fp32 results of the blocks are no further from float64."""
    import aq_mi355
    routes, E, few, N = 2600, 80, 8, 1280
    say("error of blocks of routes", gs, K)
    rng = np.random.default_rng(K)
    words, s, b = F.synthetic_affine(E * N, K, 4, gs, seed=K)
    x = F.synthetic_x(routes // 2, K, seed=5)
    rhs, lhs = rng.integers(0, E, routes).astype(np.int32), rng.integers(0, routes // 2, routes).astype(np.int32)
    mine = np.nonzero(rhs < few)[0]
    dw, dx = DeviceAffine(ctx, words, s, b), ctx.to_device(x)

    def run(ids, rows, experts):
        dr, dl, dy = ctx.to_device(ids), ctx.to_device(rows), ctx.alloc(len(ids) * N * 4)
        ctx.gather_qmv(dx, dw.w, dw.s, dw.b, dl, dr, dy, len(ids), routes // 2, K, N, experts, N, 0, gs, 4, aq_mi355.AQ_OUT_F32)
        ctx.sync()
        got = dy.download(np.float32, len(ids) * N).reshape(len(ids), N).astype(np.float64)
        for t in (dr, dl, dy):
            t.free()
        return got, ctx.last_variant(0)

    blocks, name = run(rhs, lhs, E)
    assert name == "gather_grouped_blocks", name
    tiles, name = run(rhs[mine], lhs[mine], few)
    assert name == "gather_grouped_tiles", name
    ref = np.zeros_like(tiles)
    for e in range(few):
        z, rows = np.nonzero(rhs[mine] == e)[0], slice(e * N, (e + 1) * N)
        ref[z] = F.reference_f64(x[lhs[mine][z]], words[rows], s[rows], b[rows], 4, gs, K)
    assert np.linalg.norm(blocks[mine] - ref) <= np.linalg.norm(tiles - ref)
    for t in (dx, dw):
        t.free()
