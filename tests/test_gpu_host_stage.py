"""The entry points over host slices: the staged upload gives the bytes of the same call on resident tensors, from one piece
to more than the pinned ring holds, from several threads at once, and fp32 activations round as the reference's codec does."""
import threading

import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, run_qmv, say

pytestmark = pytest.mark.gpu


# one copy by the caller; just beyond it; a few runs; the last piece short; beyond the ring of 64 MiB; a result beyond the
# pinned block of 16 MiB
@pytest.mark.parametrize("M,K,N,bits,gs", [(1, 64, 8, 4, 64), (1, 1024, 700, 4, 64), (3, 1024, 800, 4, 32), (1, 4096, 4096, 8, 64), (70, 2048, 3001, 4, 64),
                                           (1, 4096, 33000, 4, 64), (300, 64, 33001, 4, 64)])
def test_staged_call_has_the_bytes_of_the_resident_call(ctx, M, K, N, bits, gs):
    say("host slices", M, K, N, bits, gs)
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=3000 + N)
    rng = np.random.default_rng(N)
    xf = rng.normal(0, 1, (M, K)).astype(np.float32)
    xf[0, :4] = (1.00390625, 1.01171875, -1.00390625, 0.0)  # ties of the rounding to bf16
    xb = F.f32_to_bf16_bits(xf).reshape(M, K)
    dw = DeviceAffine(ctx, words, s, b)
    want = run_qmv(ctx, xb, dw, M, K, N, gs, bits, False, fn="qmv" if M == 1 else "qmm").reshape(M, N)
    for _ in range(2):
        got = ctx.proj_quant_matmul_host(xf, words, s, b, M, K, N, gs, bits)
        assert np.array_equal(F.f32_to_bf16_bits(got).reshape(M, N), want)
        if M == 1:
            assert np.array_equal(ctx.matvec_host(xb, words, s, b, N, K, gs, bits).view(np.uint16), want[0])
    dw.free()


def test_staged_calls_from_several_threads(ctx):
    say("host slices, threads")
    K, shapes = 2048, (500, 3000, 9000)
    jobs = []
    for i, N in enumerate(shapes):
        words, s, b = F.synthetic_affine(N, K, 4, 64, seed=3100 + i)
        x = F.synthetic_x(1, K, seed=3150 + i)
        jobs.append((N, words, s, b, x, ctx.matvec_host(x, words, s, b, N, K, 64, 4)))
    wrong = []

    def run(job):
        N, words, s, b, x, want = job
        for _ in range(20):
            if not np.array_equal(ctx.matvec_host(x, words, s, b, N, K, 64, 4), want):
                wrong.append(N)

    threads = [threading.Thread(target=run, args=(j,)) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_nan_activations_stay_nan(ctx):
    say("host slices, NaN")
    K, N = 64, 8
    words, s, b = F.synthetic_affine(N, K, 4, 64, seed=3200)
    x = np.zeros((2, K), np.float32)
    x[0, 5] = np.float32(np.nan)
    x[0, 6] = np.frombuffer(np.uint32(0x7f800001).tobytes(), np.float32)[0]  # a signalling NaN whose high half alone would be infinity
    x[1, 0] = 1.0
    y = ctx.proj_quant_matmul_host(x, words, s, b, 2, K, N, 64, 4)
    assert np.isnan(y[0]).all() and np.isfinite(y[1]).all()


def test_kept_device_block_is_counted():
    import aq_mi355
    say("host slices, bytes held")
    c = aq_mi355.Context(0)
    try:
        K, held = 2048, [c.workspace_bytes()]
        for N in (512, 4096, 100):
            words, s, b = F.synthetic_affine(N, K, 4, 64, seed=3300 + N)
            c.matvec_host(F.synthetic_x(1, K, seed=3301), words, s, b, N, K, 64, 4)
            held.append(c.workspace_bytes())
        assert held[1] - held[0] >= 512 * K // 2 and held[2] - held[0] >= 4096 * K // 2 and held[3] == held[2]
    finally:
        c.close()
