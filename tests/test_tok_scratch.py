"""Calls that keep rows of their own in the context's workspace while a matvec runs (the gated down projection, heads of several
rows, tile-major weights) put them behind qmm_scratch_bytes: the partial tiles of the token-tile kernels stay inside it."""
import ctypes
import os
import random

import pytest

_SO = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "go-inference_amd", "libaq_mi355.so")


@pytest.fixture(scope="module")
def lib():
    so = ctypes.CDLL(_SO)
    region, split, tiles = so._ZN2aq17qmm_scratch_bytesEiiii, so._ZN2aq10qmvt_splitEiiiiibiPiS0_, so._ZN2aq15qmvt_tile_bytesEiibi
    region.argtypes, region.restype = [ctypes.c_int] * 4, ctypes.c_size_t
    split.argtypes, split.restype = [ctypes.c_int] * 5 + [ctypes.c_bool, ctypes.c_int, ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_int)], None
    tiles.argtypes, tiles.restype = [ctypes.c_int, ctypes.c_int, ctypes.c_bool, ctypes.c_int], ctypes.c_size_t
    return region, split, tiles


@pytest.mark.parametrize("cus", [256, 128, 512])
def test_partial_tiles_stay_inside_the_region(lib, cus):
    region, split, tiles = lib
    rng = random.Random(cus)
    shapes = [(M, K, N) for M in (1, 2, 3, 4, 5, 32, 33, 64) for K in (64, 4096, 14336, 16384) for N in (1, 528, 2560, 7168, 28672, 262144)]
    shapes += [(rng.randint(1, 64), 64 * rng.randint(1, 256), int(2 ** rng.uniform(0, 18))) for _ in range(3000)]
    shares = 0
    for M, K, N in shapes:
        have = region(M, K, N, cus)
        for bits in (4, 8):
            for group in (32, 64, 128):
                k, s = ctypes.c_int(), ctypes.c_int()
                for pair in (False, True):
                    split(bits, group, M, K, N, pair, cus, ctypes.byref(k), ctypes.byref(s))
                    assert k.value == 1 or (k.value - 1) * s.value < (K + 255) // 256 <= k.value * s.value
                    shares += k.value > 1
                    assert tiles(M, N, pair, k.value) <= (2 * have if pair else have), (M, K, N, bits, group, pair)  # (pairs keep two)
    assert shares > 1000
