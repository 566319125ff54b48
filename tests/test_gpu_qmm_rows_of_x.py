"""The pass over x ahead of the fp16 matmul kernels, where its workgroups change: rows of x a workgroup, one or several passes over
a row, rows that end inside a block of 32, rows of zeros, of large and small values, of infinities and NaN."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, run_qmv, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,gs,M,K", [(4, 32, 33, 64), (4, 32, 256, 4096), (8, 32, 257, 4160), (4, 32, 257, 16448), (8, 32, 290, 960), (4, 32, 70, 32832),
                                         (4, 128, 1535, 640), (4, 64, 1536, 4096), (8, 64, 1541, 704), (4, 32, 1601, 192), (4, 64, 1540, 4160)])
def test_rows(ctx, bits, gs, M, K):
    N = 70
    say("qmm rows of x", bits, gs, M, K)
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=2800 + K)
    x = F.synthetic_x(M, K, seed=2801 + M).reshape(M, K).copy()
    f = F.bf16_bits_to_f32(x).reshape(M, K)
    f[1] *= 2.0 ** 60
    f[3] *= 2.0 ** -60
    f[5] = 0.0
    f[7, : K - 1] = 0.0
    x = F.f32_to_bf16_bits(f).reshape(M, K)
    odd = [M - 1, 9]
    x[M - 1, K - 1] = 0x7F80  # inf
    x[9, 0] = 0xFFC0          # NaN
    dw = DeviceAffine(ctx, words, s, b)
    got = run_qmv(ctx, x, dw, M, K, N, gs, bits, True, fn="qmm").reshape(M, N).astype(np.float64)
    assert ctx.last_variant(1).startswith("qmmh"), ctx.last_variant(1)
    assert not np.isfinite(got[odd]).any()
    rows = [r for r in (0, 1, 2, 3, 5, 7, 8, 15, 16, 31, 32, M // 2, M - 3, M - 2) if r < M - 1]
    ref = F.reference_f64(x[rows], words, s, b, bits, gs, K)
    # K / 16 steps of the matrix cores, each a rounding of 2^-24 of the sum so far, as a random walk: sqrt(32832 / 16) = 45 < 2^6
    assert (np.linalg.norm(got[rows] - ref, axis=1) <= 2.0 ** -18 * np.linalg.norm(ref, axis=1)).all()
    assert np.isfinite(np.delete(got, odd, axis=0)).all()
    dw.free()
