"""The fp16-operand matmul kernels on 8-bit codes: every tile, groups of 32, 64 and 128, K shared out over workgroups, several
matrices in one grid, the gated pair, expert slabs.  Accumulators within the stated bounds of the float64 reference."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, run_qmv, say

pytestmark = pytest.mark.gpu

# edges of 32-, 64- and 128-row tiles; K of one block, a piece of a quad, shares of K of which the last is short
SHAPES = [(32, 5, 64, 40), (32, 33, 192, 257), (32, 64, 4032, 70), (64, 65, 1088, 1001), (128, 129, 640, 300), (32, 509, 960, 2050), (64, 200, 3840, 8200),
          (64, 777, 2560, 512), (128, 66, 512, 33), (64, 1030, 512, 4100)]


@pytest.mark.parametrize("gs,M,K,N", SHAPES)
def test_shapes(ctx, gs, M, K, N):
    say("qmm 8 bit", gs, M, K, N)
    words, s, b = F.synthetic_affine(N, K, 8, gs, seed=3400 + M)
    x = F.synthetic_x(M, K, seed=3401 + K)
    dw = DeviceAffine(ctx, words, s, b)
    acc = run_qmv(ctx, x, dw, M, K, N, gs, 8, True, fn="qmm")
    name = ctx.last_variant(1)
    assert name.startswith("qmmh8_b8_"), name
    cols = np.unique(np.r_[0, N - 1, np.random.default_rng(7).choice(N, min(N, 160), replace=False)])
    check_accumulators(acc[:, cols], F.reference_f64(x, words[cols], s[cols], b[cols], 8, gs, K), "%s M=%d K=%d N=%d" % (name, M, K, N))
    out = run_qmv(ctx, x, dw, M, K, N, gs, 8, False, fn="qmm")
    assert np.array_equal(out, F.f32_to_bf16_bits(acc).reshape(M, N))
    dw.free()


@pytest.mark.parametrize("M,K,N", [(31, 64, 33), (97, 192, 260), (300, 704, 515)])
def test_every_tile(ctx, M, K, N):
    """Each tile on shapes that end inside it; which tile runs does not show in the bytes."""
    import aq_mi355
    words, s, b = F.synthetic_affine(N, K, 8, 64, seed=3450)
    x = F.synthetic_x(M, K, seed=3451)
    dw = DeviceAffine(ctx, words, s, b)
    ref, first = F.reference_f64(x, words, s, b, 8, 64, K), None
    for i, name in enumerate(aq_mi355.variant_names(1)):
        if not name.startswith("qmmh8_b8_"):
            continue
        say("qmm 8 bit tile", name, M, K, N)
        ctx.force_variant(1, i)
        try:
            acc = run_qmv(ctx, x, dw, M, K, N, 64, 8, True, fn="qmm")
        finally:
            ctx.force_variant(1, -1)
        check_accumulators(acc, ref, name)
        first = acc if first is None else first
        assert np.array_equal(acc.view(np.uint32), first.view(np.uint32)), name
    assert first is not None
    dw.free()


@pytest.mark.parametrize("gs,M,K,Ns", [(32, 70, 1024, (256, 64, 64)), (64, 300, 4096, (1024, 130, 256)), (128, 100, 2048, (512, 300))])
def test_matrices_in_one_grid_have_the_bytes_of_their_own_calls(ctx, gs, M, K, Ns):
    import aq_mi355
    say("qmm 8 bit multi", gs, M, K, Ns)
    mats = [F.synthetic_affine(n, K, 8, gs, seed=3500 + i) for i, n in enumerate(Ns)]
    x = F.synthetic_x(M, K, seed=3550)
    dws = [DeviceAffine(ctx, *m) for m in mats]
    alone = [run_qmv(ctx, x, d, M, K, n, gs, 8, True, fn="qmm") for d, n in zip(dws, Ns)]
    dx, ys = ctx.to_device(x), [ctx.alloc(M * n * 4) for n in Ns]
    ctx.qmm_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, 8, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    for n, y, one in zip(Ns, ys, alone):
        assert np.array_equal(y.download(np.uint32, M * n).reshape(M, n), one.reshape(M, n).view(np.uint32))
    for t in [dx] + ys + dws:
        t.free()


@pytest.mark.parametrize("gs,M,K,N", [(32, 33, 960, 130), (32, 509, 1024, 515), (64, 65, 4096, 512), (128, 300, 2048, 264)])
def test_gated_pair(ctx, orc, gs, M, K, N):
    import aq_mi355
    say("qmm 8 bit gate|up", gs, M, K, N)
    gate, up = F.synthetic_affine(N, K, 8, gs, seed=3600), F.synthetic_affine(N, K, 8, gs, seed=3601)
    x = F.synthetic_x(M, K, seed=3602)
    dg, du = DeviceAffine(ctx, *gate), DeviceAffine(ctx, *up)
    g, u = (run_qmv(ctx, x, d, M, K, N, gs, 8, True, fn="qmm").reshape(M, N) for d in (dg, du))
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    act = aq_mi355.AQ_ACT_GELU_TANH
    ctx.qmv_gate_up(dx, (dg.w, dg.s, dg.b), (du.w, du.s, du.b), dy, M, K, N, gs, 8, act, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0) == "qmv_gate_up_tiles" and ctx.last_variant(1).startswith("qmmh8_b8_")
    got = dy.download(np.float32, M * N).reshape(M, N)
    want = orc.act_multiply(act, g.reshape(-1), u.reshape(-1)).reshape(M, N)
    # the same fp32 sums; tanh of the device library against the oracle's: a few fp32 ulp
    assert (np.abs(got - want) <= 4e-6 * np.abs(want) + 2.5e-7 * np.maximum(1.0, np.abs(g * u))).all()
    for t in (dx, dy, dg, du):
        t.free()
