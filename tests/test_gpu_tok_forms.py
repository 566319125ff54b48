"""The token-tile kernels beyond groups of 64 with whole runs of 256 codes: groups of 32 and 128, a K that ends inside a
run, several matrices in one grid and the gated pair.  Accumulators within the stated bounds of the float64 reference."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, check_bf16_store, run_qmv, say

pytestmark = pytest.mark.gpu

# K: one piece of a run, a run and a piece, every number of 64-code blocks in the last run, one run per wavefront and more
SHAPES = [(bits, 32, M, K, N) for bits in (4, 8) for M, K, N in ((3, 64, 40), (16, 192, 1030), (17, 320, 70), (32, 4096, 16), (9, 4032, 130))]
SHAPES += [(bits, 128, M, K, N) for bits in (4, 8) for M, K, N in ((5, 128, 33), (16, 2944, 66), (32, 4096, 49))]
SHAPES += [(bits, 64, M, K, N) for bits in (4, 8) for M, K, N in ((9, 960, 4400), (16, 2112, 2001), (32, 4032, 1056))]
# small matrices with such a K, from the first size that runs here
SHAPES += [(4, 64, 9, 320, 529), (4, 64, 32, 4160, 600), (8, 64, 5, 64, 1), (8, 64, 5, 320, 24), (8, 64, 32, 4160, 48)]


@pytest.mark.parametrize("bits,gs,M,K,N", SHAPES)
def test_token_tile_forms(ctx, bits, gs, M, K, N):
    say("token tile", bits, gs, M, K, N)
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=2100 + K)
    x = F.synthetic_x(M, K, seed=2101 + M)
    ref = F.reference_f64(x, words, s, b, bits, gs, K)
    dw = DeviceAffine(ctx, words, s, b)
    acc = run_qmv(ctx, x, dw, M, K, N, gs, bits, True)
    name = ctx.last_variant(0)
    exact = gs == 64 and K % 256 == 0
    assert name.startswith("qmvt_b%d_" % bits) and name.endswith("_s32" if gs == 32 else "_d2" if exact else "_any"), name
    check_accumulators(acc, ref, name)
    out = run_qmv(ctx, x, dw, M, K, N, gs, bits, False)
    assert np.array_equal(out, F.f32_to_bf16_bits(acc).reshape(M, N))
    dw.free()


@pytest.mark.parametrize("bits,gs,M,K,Ns", [(4, 64, 12, 4032, (1056, 200, 17)), (4, 32, 4, 3840, (130, 64, 1)), (8, 64, 20, 2048, (512, 96)),
                                            (8, 32, 2, 960, (40, 50, 60, 70)), (4, 128, 32, 1024, (256, 300))])
def test_several_matrices_in_one_grid(ctx, bits, gs, M, K, Ns):
    say("token tile multi", bits, gs, M, K, Ns)
    mats = [F.synthetic_affine(n, K, bits, gs, seed=2200 + i) for i, n in enumerate(Ns)]
    x = F.synthetic_x(M, K, seed=2250)
    dws = [DeviceAffine(ctx, *m) for m in mats]
    dx, ys = ctx.to_device(x), [ctx.alloc(M * n * 2) for n in Ns]
    ctx.qmv_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, bits)
    ctx.sync()
    assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
    for n, m, y in zip(Ns, mats, ys):
        check_bf16_store(y.download(np.uint16, M * n), F.reference_f64(x, *m, bits, gs, K), "member of %d rows" % n)
    for t in [dx] + ys + dws:
        t.free()


@pytest.mark.parametrize("bits,gs,M,K,N", [(4, 32, 21, 3840, 1000), (4, 64, 9, 4096, 77), (8, 64, 32, 960, 4400), (8, 32, 2, 192, 33),
                                           (4, 128, 16, 640, 48)])
def test_gated_pair(ctx, orc, bits, gs, M, K, N):
    """act(gate . x) * (up . x) in one launch from the sums of the separate projections."""
    say("token tile gate|up", bits, gs, M, K, N)
    gate, up = F.synthetic_affine(N, K, bits, gs, seed=2300), F.synthetic_affine(N, K, bits, gs, seed=2301)
    x = F.synthetic_x(M, K, seed=2302)
    dg, du = DeviceAffine(ctx, *gate), DeviceAffine(ctx, *up)
    g = run_qmv(ctx, x, dg, M, K, N, gs, bits, True)
    u = run_qmv(ctx, x, du, M, K, N, gs, bits, True)
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    import aq_mi355
    for act in (aq_mi355.AQ_ACT_GELU_TANH, aq_mi355.AQ_ACT_SILU):
        ctx.qmv_gate_up(dx, (dg.w, dg.s, dg.b), (du.w, du.s, du.b), dy, M, K, N, gs, bits, act, aq_mi355.AQ_OUT_F32)
        ctx.sync()
        assert ctx.last_variant(0) == "qmv_gate_up_tok"
        got = dy.download(np.float32, M * N).reshape(M, N)
        want = orc.act_multiply(act, g, u)
        # the same fp32 sums; tanh and exp of the device library against the oracle's: a few fp32 ulp
        assert (np.abs(got - want) <= 4e-6 * np.abs(want) + 2.5e-7 * np.maximum(1.0, np.abs(g * u))).all()
    for t in (dx, dy, dg, du):
        t.free()


@pytest.mark.parametrize("bits,gs,M,K", [(4, 64, 9, 4096), (8, 64, 2, 4096), (4, 32, 3, 960), (4, 128, 32, 1024), (4, 64, 1, 4096), (4, 64, 48, 4096)])
def test_several_matrices_without_x_are_refused(ctx, bits, gs, M, K):
    import aq_mi355
    say("token tile multi without x", bits, gs, M, K)
    dws, ys = [], []
    for n in (48, 16):
        dws.append(DeviceAffine(ctx, *F.synthetic_affine(n, K, bits, gs, seed=2260)))
        ys.append(ctx.alloc(M * n * 2))
    with pytest.raises(aq_mi355.AqError) as e:
        ctx.qmv_multi(None, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, [48, 16], M, K, gs, bits)
    assert e.value.code == aq_mi355.AQ_ERR_ARG and "null operand" in str(e.value)
    ctx.sync()
    for t in ys + dws:
        t.free()


# the sum of the rows on one side of a line of the selection and every member on the other (40 Mi and 4 Mi codes), members on
# both sides of it, and shapes without such a line
@pytest.mark.parametrize("bits,gs,M,K,Ns", [(8, 64, 2, 4096, (4096, 4096, 4096)), (8, 64, 4, 8192, (2048, 3100, 512)), (8, 64, 2, 2112, (900, 1100, 400)),
                                            (8, 64, 8, 4032, (520, 520, 600)), (4, 64, 12, 4032, (520, 520, 600)), (4, 64, 32, 2112, (2100, 300)),
                                            (4, 64, 6, 4032, (520, 600)), (4, 32, 5, 3840, (130, 64, 1)), (8, 32, 2, 960, (40, 50)), (4, 128, 5, 1024, (256, 300)),
                                            (8, 128, 3, 1024, (256, 300)), (4, 64, 16, 4096, (1000, 17))])
def test_members_have_the_bytes_of_their_own_calls(ctx, bits, gs, M, K, Ns):
    import aq_mi355
    say("token tile multi, bytes", bits, gs, M, K, Ns)
    x = F.synthetic_x(M, K, seed=2270)
    dws = [DeviceAffine(ctx, *F.synthetic_affine(n, K, bits, gs, seed=2271 + i)) for i, n in enumerate(Ns)]
    alone = [run_qmv(ctx, x, d, M, K, n, gs, bits, True) for d, n in zip(dws, Ns)]
    dx, ys = ctx.to_device(x), [ctx.alloc(M * n * 4) for n in Ns]
    ctx.qmv_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, gs, bits, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    for n, y, one in zip(Ns, ys, alone):
        assert np.array_equal(y.download(np.uint32, M * n), one.view(np.uint32).reshape(-1)), "member of %d rows" % n
    for t in [dx] + ys + dws:
        t.free()


@pytest.mark.parametrize("off_gate,off_up,fused", [(0, 0, True), (8, 8, True), (8, 0, True), (8, 2, False), (2, 8, False), (4, 4, False)])
def test_gated_pair_scales_of_any_alignment(ctx, orc, off_gate, off_up, fused):
    """Scales and biases of the two matrices at their own byte offsets: the one launch asks the same of both, and the separate
    projections run where either falls short of it."""
    import aq_mi355
    M, K, N, gs, bits = 12, 1024, 200, 64, 4
    say("token tile gate|up, alignment", off_gate, off_up)
    x = F.synthetic_x(M, K, seed=2350)
    mats = [F.synthetic_affine(N, K, bits, gs, seed=2351 + i) for i in range(2)]
    g, u = (F.reference_f64(x, *m, bits, gs, K) for m in mats)
    held, args = [], []
    for (words, s, b), off in zip(mats, (off_gate, off_up)):
        sb = [ctx.to_device(np.concatenate([np.zeros(off // 2, np.uint16), np.ravel(t)])) for t in (s, b)]
        held += [ctx.to_device(words)] + sb
        args.append((held[-3], sb[0].ptr + off, sb[1].ptr + off))
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    ctx.qmv_gate_up(dx, args[0], args[1], dy, M, K, N, gs, bits, aq_mi355.AQ_ACT_SILU, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert (ctx.last_variant(0) == "qmv_gate_up_tok") == fused, ctx.last_variant(0)
    want = g / (1.0 + np.exp(-g)) * u
    got = dy.download(np.float32, M * N).reshape(M, N)
    # 1e-4: twice the fp32 sums' error over K = 1024 against float64 (1.2e-5 of the result's scale on the code-128 kernels)
    assert (np.abs(got - want) <= 1e-4 * np.maximum(1.0, np.abs(g * u) + np.abs(g) + np.abs(u))).all()
    for t in held + [dx, dy]:
        t.free()


@pytest.mark.parametrize("bits,gs,M,K,N", [(4, 32, 3, 3840, 300), (4, 32, 21, 3840, 300), (4, 32, 32, 1024, 300), (4, 32, 21, 15360, 64), (4, 128, 12, 2944, 300),
                                           (4, 64, 20, 4032, 1056), (8, 32, 21, 3840, 300), (8, 64, 3, 4032, 1056), (8, 128, 32, 2944, 300)])
def test_sums_keep_fp32_accuracy(ctx, bits, gs, M, K, N):
    """Weights centred on zero, as GGUF tensors and the synthetic ones are: what the operand's codes carry beside the weight
    must not be taken off again out of a sum many times the result.  2^-21 = 4.8e-7 of the result's 2-norm: eight roundings of
    2^-24 on the way (the fp32 sums of the any-width kernel end at 0.7e-7 to 2.5e-7, sums over 128 + code at 2e-6)."""
    say("token tile accuracy", bits, gs, M, K, N)
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=2390 + K)
    x = F.synthetic_x(M, K, seed=2391 + M)
    dw = DeviceAffine(ctx, words, s, b)
    got = run_qmv(ctx, x, dw, M, K, N, gs, bits, True).astype(np.float64)
    assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
    ref = F.reference_f64(x, words, s, b, bits, gs, K)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print("error %.2e" % err)
    assert err <= 2.0 ** -21
    dw.free()


@pytest.mark.parametrize("bits,gs,M,K,N", [(8, 64, 9, 64, 1), (8, 64, 17, 64, 3), (8, 64, 5, 192, 1), (4, 32, 5, 64, 1), (4, 32, 20, 64, 3), (8, 32, 9, 192, 1),
                                           (8, 32, 2, 64, 4), (4, 128, 9, 128, 3), (4, 128, 18, 384, 1), (8, 128, 6, 384, 1), (4, 128, 6, 128, 4)])
def test_matrices_of_fewer_groups_than_a_load_of_scales(ctx, bits, gs, M, K, N):
    import aq_mi355
    say("tok tiny", bits, gs, M, K, N)
    mats = [F.synthetic_affine(N, K, bits, gs, seed=2600 + K + i) for i in range(2)]
    x = F.synthetic_x(M, K, seed=2602)
    dws = [DeviceAffine(ctx, *m) for m in mats]
    acc = run_qmv(ctx, x, dws[0], M, K, N, gs, bits, True)
    assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
    g, u = (F.reference_f64(x, *m, bits, gs, K) for m in mats)
    check_accumulators(acc, g, "tiny")
    dx, dy = ctx.to_device(x), ctx.alloc(M * N * 4)
    ctx.qmv_gate_up(dx, *((d.w, d.s, d.b) for d in dws), dy, M, K, N, gs, bits, aq_mi355.AQ_ACT_SILU, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0) == "qmv_gate_up_tok"
    check_accumulators(dy.download(np.float32, M * N), g / (1.0 + np.exp(-g)) * u, "tiny pair")
    for t in [dx, dy] + dws:
        t.free()
