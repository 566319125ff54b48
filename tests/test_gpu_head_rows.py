"""Greedy tokens of several rows: the argmax over fp32 scores in memory, at the lengths where its launch changes shape (one
workgroup a row, several that meet in an atomic maximum).  The best value of a row is the maximum of its packed scores."""
import numpy as np
import pytest

import fixtures as F
from gpu_util import DeviceAffine, say
from test_gpu_head import _greedy, _scores

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(2, 1), (3, 1023), (2, 8193), (3, 16384), (2, 16385), (5, 140001)])
def test_best_of_every_row(ctx, M, N):
    say("greedy rows", M, N)
    K, gs, bits = 64, 64, 4
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=F.BASE_SEED + 110)
    words[N // 2] = words[N - 1]                    # equal rows: the lower one wins
    s[N // 2], b[N // 2] = s[N - 1], b[N - 1]
    if N > 2:
        s[1] = 0x7FC0                               # a row without a finite score
    x = F.synthetic_x(M, K, seed=F.BASE_SEED + 111)
    dw = DeviceAffine(ctx, words, s, b)
    packed = _scores(ctx, x, dw, M, K, N, gs, bits)
    assert np.array_equal(_greedy(ctx, x, dw, M, K, N, gs, bits), packed.max(axis=1))
    winners = sorted({int(p.argmax()) for p in packed} | {0, N - 1})
    packed = _scores(ctx, x, dw, M, K, N, gs, bits, winners)
    assert np.array_equal(_greedy(ctx, x, dw, M, K, N, gs, bits, winners), packed.max(axis=1))
    dw.free()


# one workgroup a row and several with the list as bits, its longest row, and the first that goes through the list
@pytest.mark.parametrize("M,N,count", [(2, 16384, 300), (3, 16385, 1100), (1, 524288, 70), (2, 524288, 70), (2, 524289, 70)])
def test_best_behind_a_long_list(ctx, M, N, count):
    say("greedy rows, suppressed", M, N, count)
    K, gs, bits = 64, 64, 4
    words, s, b = F.synthetic_affine(N, K, bits, gs, seed=F.BASE_SEED + 112)
    x = F.synthetic_x(M, K, seed=F.BASE_SEED + 113)
    dw = DeviceAffine(ctx, words, s, b)
    packed = _scores(ctx, x, dw, M, K, N, gs, bits)
    gone = np.unique(np.concatenate([np.argsort(p)[::-1][:count] for p in packed] + [[0, N - 1]]))
    listed = list(map(int, gone)) + [-1, N, N + 5, int(gone[0])]   # tokens that there are not, one twice
    packed[:, gone] = 0
    assert np.array_equal(_greedy(ctx, x, dw, M, K, N, gs, bits, listed), packed.max(axis=1))
    dw.free()
