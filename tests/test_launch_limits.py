"""The stateless operators' choice of kernel, asked without a GPU: a launch
holds at most 2^32 - 1 threads along x (HIP refuses more), so no call may be
given a kernel whose grid is larger, and every call that 128-row tiles hold
must be given one.  Operand pointers serve for their alignment only."""

import ctypes as C

import pytest

import bfhip

LIMIT = 2 ** 32 - 1
# GemmRoute of ops.hip: rows x columns of a workgroup's tile, threads.
GEMM_TILES = {0: (128, 128, 512), 1: (64, 64, 256), 2: (32, 32, 256), 3: (16, 16, 512),
              4: (64, 16, 256), 5: (128, 128, 256), 6: (128, 1 << 30, 512)}


def _threads(m, n, tile):
    bm, bn, threads = tile
    return -(-m // bm) * -(-n // bn) * threads


def gemm_route(m, k, n, aligned=True):
    f = bfhip.hip_lib().bfhip_gemm_route
    f.argtypes = [C.c_void_p] * 4 + [C.c_int] * 3
    p = 4096 if aligned else 4100
    return f(p, p, None, p, m, k, n)


@pytest.mark.parametrize("n", [1, 16, 17, 32, 33, 64, 65, 129, 148, 288, 300, 4096, 1048560])
def test_gemm_grids_fit_a_launch(n):
    tile = (128, 32, 256) if n <= 32 else (128, 64, 256) if n <= 64 else (128, 128, 256)
    rows = {1, 127, 10 ** 6, 2 ** 31 - 1}
    for bits in range(20, 32):
        rows |= {2 ** bits + d for d in (-129, -1, 0, 1, 77, 2 ** (bits - 1)) if 2 ** bits + d < 2 ** 31}
    for m in sorted(rows):
        for k in (1, 8, 100, 130, 3072):
            for aligned in (True, False):
                route = gemm_route(m, k, n, aligned)
                if route >= 0 and route != 6:
                    assert _threads(m, n, GEMM_TILES[route]) <= LIMIT, (m, k, n, route)
                if _threads(m, n, tile) <= LIMIT:
                    assert route >= 0, (m, k, n)


def test_gemm_route_of_very_many_rows():
    """2^30 rows and a few: the thin and 64-row tiles no longer fit."""
    assert gemm_route(2 ** 30 + 77, 1, 1) == 5
