"""Dense calls in groups of 32 with infinities and NaN in x: every output is what the sum over fp32 weights makes of them (an
infinity by the sign of its weight, NaN where signs meet or the weight is zero), on every kernel that takes such calls, and
other rows are as without them."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, check_accumulators, run_qmv, say

pytestmark = pytest.mark.gpu


def _inputs(M, K, N, bits, seed):
    words, s, b = F.synthetic_affine(N, K, bits, 32, seed=seed)
    x = F.f32_to_bf16_bits(F.bf16_bits_to_f32(F.synthetic_x(M, K, seed=seed + 1))).reshape(M, K)
    odd = x.copy()
    inf = np.uint16(0x7f80)
    odd[0, 5] = inf                               # one of either sign, in the first and the last group
    odd[2, K - 1] = inf | 0x8000
    odd[1, 7], odd[1, K // 2] = inf, inf | 0x8000  # two that may meet
    odd[M - 1, 3] = 0x7fc0                        # NaN
    return words, s, b, x, odd


def _expected(odd, words, s, b, bits, K):
    w = F.numpy_dequant(words, s, b, bits, 32, K)
    xf = F.bf16_bits_to_f32(odd)
    with np.errstate(invalid="ignore"):
        return np.array([[(xf[m, ~np.isfinite(xf[m])] * w[n, ~np.isfinite(xf[m])]).sum() for n in range(w.shape[0])] for m in (0, 1, 2, -1)])


def _check(got, want, odd, words, s, b, bits, K):
    rows = [0, 1, 2, odd.shape[0] - 1]
    assert np.array_equal(got[rows], want, equal_nan=True)
    rest = np.setdiff1d(np.arange(odd.shape[0]), rows)
    if rest.size:
        check_accumulators(got[rest], F.reference_f64(odd[rest], words, s, b, bits, 32, K), "rows without infinities")


@pytest.mark.parametrize("fn,M,K,N", [("qmv", 5, 960, 70), ("qmv", 21, 3840, 90), ("qmv", 32, 192, 33), ("qmm", 7, 960, 40), ("qmm", 40, 4096, 130),
                                      ("qmm", 130, 512, 600), ("qmm", 300, 192, 1100)])
@pytest.mark.parametrize("bits", [4, 8])
def test_projection(ctx, bits, fn, M, K, N):
    say("infinities", bits, fn, M, K, N)
    words, s, b, x, odd = _inputs(M, K, N, bits, 3300 + M)
    dw = DeviceAffine(ctx, words, s, b)
    got = run_qmv(ctx, odd, dw, M, K, N, 32, bits, True, fn=fn).reshape(M, N)
    name = ctx.last_variant(0 if fn == "qmv" else 1)
    assert name.startswith("qmvt_" if fn == "qmv" else "qmmh"), name
    _check(got, _expected(odd, words, s, b, bits, K), odd, words, s, b, bits, K)
    out = run_qmv(ctx, odd, dw, M, K, N, 32, bits, False, fn=fn)
    assert np.array_equal(F.bf16_bits_to_f32(out).reshape(M, N), F.bf16_bits_to_f32(F.f32_to_bf16_bits(got)).reshape(M, N), equal_nan=True)
    base = run_qmv(ctx, x, dw, M, K, N, 32, bits, True, fn=fn).reshape(M, N)
    rest = np.setdiff1d(np.arange(M), [0, 1, 2, M - 1])
    assert np.array_equal(got[rest].view(np.uint32), base[rest].view(np.uint32))
    dw.free()


def test_products_beyond_fp32_of_the_codes_alone(ctx):
    """x near the end of bf16's range against small weights: the outputs are finite though codes times x are not."""
    M, K, N = 20, 256, 40
    say("infinities, large x")
    words, s, b = F.synthetic_affine(N, K, 4, 32, seed=3390)
    scaled = lambda t, p: F.f32_to_bf16_bits((F.bf16_bits_to_f32(t) * np.float32(2.0 ** p)).astype(np.float32)).reshape(t.shape)
    x, s, b = scaled(F.synthetic_x(M, K, seed=3391), 123), scaled(s, -30), scaled(b, -30)
    ref = F.reference_f64(x, words, s, b, 4, 32, K)
    dw = DeviceAffine(ctx, words, s, b)
    for fn in ("qmv", "qmm"):
        got = run_qmv(ctx, x, dw, M, K, N, 32, 4, True, fn=fn).reshape(M, N).astype(np.float64)
        assert np.isfinite(got).all()
        assert np.linalg.norm((got - ref) / 2.0 ** 93) <= 2.0 ** -21 * np.linalg.norm(ref / 2.0 ** 93), fn
    dw.free()


@pytest.mark.parametrize("M,K,N", [(21, 960, 70), (40, 4096, 130), (130, 512, 600)])
@pytest.mark.parametrize("bits", [4, 8])
def test_gated_pair(ctx, orc, bits, M, K, N):
    import aq_mi355
    say("infinities, gate|up", bits, M, K, N)
    gw, gs, gb, x, odd = _inputs(M, K, N, bits, 3400 + M)
    uw, us, ub = F.synthetic_affine(N, K, bits, 32, seed=3450)
    dg, du = DeviceAffine(ctx, gw, gs, gb), DeviceAffine(ctx, uw, us, ub)
    dx, dy = ctx.to_device(odd), ctx.alloc(M * N * 4)
    ctx.qmv_gate_up(dx, (dg.w, dg.s, dg.b), (du.w, du.s, du.b), dy, M, K, N, 32, bits, aq_mi355.AQ_ACT_SILU, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0) in ("qmv_gate_up_tok", "qmv_gate_up_tiles")
    got = dy.download(np.float32, M * N).reshape(M, N)
    g, u = _expected(odd, gw, gs, gb, bits, K), _expected(odd, uw, us, ub, bits, K)
    with np.errstate(all="ignore"):
        want = (g / (np.float32(1.0) + np.exp(-g)) * u).astype(np.float32)
    assert np.array_equal(got[[0, 1, 2, M - 1]], want, equal_nan=True)
    assert np.isfinite(got[3:M - 1]).all()
    for t in (dx, dy, dg, du):
        t.free()


# Calls that share K out (tests/calls_on_host.cc states that these do), whose sums meet in a launch of their own, and calls of 33..64
# rows, which run as two halves: by fours of columns and one by one, the second matrix of a pair, a member behind the first.
def _odd_halves(x, K):
    """Infinities and NaN in rows of either half; the rows that have them."""
    M, inf = x.shape[0], np.uint16(0x7f80)
    odd = x.copy()
    half = M // 2 if M > 32 else 4
    odd[0, 5], odd[2, K - 1], odd[half, K // 2 + 3], odd[M - 2, 70] = inf, inf | 0x8000, inf | 0x8000, inf
    odd[1, 7], odd[1, K // 2] = inf, inf | 0x8000
    odd[half + 1, K - 40], odd[half + 1, 40] = inf, inf | 0x8000
    odd[M - 1, 3] = 0x7fc0
    return odd, [0, 1, 2, half, half + 1, M - 2, M - 1]


def _sums(odd, rows, words, s, b, bits, K):
    w, xf = F.numpy_dequant(words, s, b, bits, 32, K), F.bf16_bits_to_f32(odd)
    with np.errstate(invalid="ignore"):
        return np.array([(w[:, ~np.isfinite(xf[m])] * xf[m, ~np.isfinite(xf[m])]).sum(axis=1) for m in rows])


@pytest.mark.parametrize("M,K,N", [(21, 15360, 100), (21, 15360, 101), (40, 2112, 600), (40, 15360, 600), (63, 15360, 545)])
@pytest.mark.parametrize("bits", [4, 8])
def test_projection_in_shares(ctx, bits, M, K, N):
    say("infinities, shares of K", bits, M, K, N)
    words, s, b = F.synthetic_affine(N, K, bits, 32, seed=3500 + M)
    x = F.synthetic_x(M, K, seed=3501).reshape(M, K)
    odd, rows = _odd_halves(x, K)
    rest = np.setdiff1d(np.arange(M), rows)
    dw = DeviceAffine(ctx, words, s, b)
    got = run_qmv(ctx, odd, dw, M, K, N, 32, bits, True)
    assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
    assert np.array_equal(got[rows], _sums(odd, rows, words, s, b, bits, K), equal_nan=True)
    base = run_qmv(ctx, x, dw, M, K, N, 32, bits, True)
    assert np.array_equal(got[rest].view(np.uint32), base[rest].view(np.uint32))
    check_accumulators(base, F.reference_f64(x, words, s, b, bits, 32, K), "without infinities")
    dw.free()


@pytest.mark.parametrize("M,K,N", [(21, 15360, 100), (21, 15360, 101), (40, 2112, 600), (40, 15360, 600)])
@pytest.mark.parametrize("bits", [4, 8])
def test_gated_pair_in_shares(ctx, bits, M, K, N):
    import aq_mi355
    say("infinities, gate|up, shares of K", bits, M, K, N)
    mats = [F.synthetic_affine(N, K, bits, 32, seed=3520 + i) for i in range(2)]
    odd, rows = _odd_halves(F.synthetic_x(M, K, seed=3522).reshape(M, K), K)
    dws = [DeviceAffine(ctx, *m) for m in mats]
    dx, dy = ctx.to_device(odd), ctx.alloc(M * N * 4)
    ctx.qmv_gate_up(dx, *((d.w, d.s, d.b) for d in dws), dy, M, K, N, 32, bits, aq_mi355.AQ_ACT_SILU, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0) == "qmv_gate_up_tok"
    got = dy.download(np.float32, M * N).reshape(M, N)
    g, u = (_sums(odd, rows, *m, bits, K) for m in mats)
    with np.errstate(all="ignore"):
        want = (g / (np.float32(1.0) + np.exp(-g)) * u).astype(np.float32)
    assert np.array_equal(got[rows], want, equal_nan=True)
    assert np.isfinite(got[np.setdiff1d(np.arange(M), rows)]).all()
    for t in [dx, dy] + dws:
        t.free()


@pytest.mark.parametrize("M,K,Ns", [(21, 5120, (12000, 100, 64)), (40, 5120, (6000, 600)), (21, 15360, (130, 65, 1)), (21, 5376, (4096, 2048, 2048))])
@pytest.mark.parametrize("bits", [4, 8])
def test_members_in_shares(ctx, bits, M, K, Ns):
    import aq_mi355
    say("infinities, members, shares of K", bits, M, K, Ns)
    mats = [F.synthetic_affine(n, K, bits, 32, seed=3540 + i) for i, n in enumerate(Ns)]
    odd, rows = _odd_halves(F.synthetic_x(M, K, seed=3543).reshape(M, K), K)
    dws = [DeviceAffine(ctx, *m) for m in mats]
    dx, ys = ctx.to_device(odd), [ctx.alloc(M * n * 4) for n in Ns]
    ctx.qmv_multi(dx, [d.w for d in dws], [d.s for d in dws], [d.b for d in dws], ys, list(Ns), M, K, 32, bits, aq_mi355.AQ_OUT_F32)
    ctx.sync()
    assert ctx.last_variant(0).startswith("qmvt_"), ctx.last_variant(0)
    for n, m, y in zip(Ns, mats, ys):
        got = y.download(np.float32, M * n).reshape(M, n)
        assert np.array_equal(got[rows], _sums(odd, rows, *m, bits, K), equal_nan=True), "member of %d rows" % n
        assert np.isfinite(got[np.setdiff1d(np.arange(M), rows)]).all()
    for t in [dx] + ys + dws:
        t.free()
