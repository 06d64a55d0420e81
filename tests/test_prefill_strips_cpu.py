"""The cut of the exact strips' work (krasis_amd/csrc/kr_prefill_strip.inc), on the host: whatever number of tiles there is, every column block of every tile has one workgroup of the grid."""
import ctypes as C
import random

import numpy as np
import pytest


def plan(strip, N, K, most, tiles):
    """(strips a wave of the first tiles, of the others, how many the first ones are), [grid, 3] of tile, column block and strips a wave"""
    from krasis_amd._lib import check, load_library
    lib = load_library()
    cut, grid = (C.c_int * 3)(), C.c_int()
    check(lib.kr_moe_strip_plan(strip, N, K, most, tiles, cut, None, 0, C.byref(grid)))
    places = np.empty((grid.value, 3), np.int32)
    check(lib.kr_moe_strip_plan(strip, N, K, most, tiles, cut, places.ctypes.data, len(places), C.byref(grid)))
    places[:, 2] = 1 << places[:, 2]
    return (1 << cut[0], 1 << cut[1], cut[2]), places


def check_plan(strip, N, K, most, tiles):
    (first, others, whole), places = plan(strip, N, K, most, tiles)
    groups = -(-(N // 16) // (8 if strip == 16 else 16))
    want = sorted((t, b, n) for t in range(tiles) for n in [first if t < whole else others] for b in range(-(-groups // n)))
    got = sorted(map(tuple, places[places[:, 0] >= 0].tolist()))
    assert got == want, (strip, N, K, most, tiles)
    return len(places)


def test_every_column_block_once():
    rng = random.Random(5)
    for _ in range(1500):
        most = rng.choice([rng.randint(1, 40), rng.randint(1, 700), rng.randint(1, 2100)])
        check_plan(rng.choice([16, 32]), 16 * rng.randint(1, 400), 128 * rng.randint(1, 24), most, rng.choice([0, 1, most, rng.randint(0, most), max(0, most - rng.randint(0, 9))]))


@pytest.mark.parametrize("strip,N,K,most,grid", [
    (16, 2048, 1408, 104, 1664),      # one strip a wave: nothing to cut, a workgroup for every column block and no more
    (16, 2816, 2048, 104, 1320),      # 88 tiles of eleven column blocks and 16 of 22
    (16, 1024, 2048, 543, 1280),      # two whole rounds of 512, and 31 tiles of eight column blocks
])
def test_no_more_workgroups_than_a_cut_needs(strip, N, K, most, grid):
    assert check_plan(strip, N, K, most, most) == grid
