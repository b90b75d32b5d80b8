"""The library's choices by size, asked on the CPU.  A launch holds at most
2^32 - 1 threads along x (HIP refuses more), so no call may be given a kernel
whose grid is larger, and every call that 128-row tiles hold must be given one;
and a choice has to be near the fastest kernel measured.  Operand pointers
serve for their alignment only."""

import ctypes as C

import pytest

import bfhip

LIMIT = 2 ** 32 - 1
# GemmRoute of ops.hip: rows x columns of a workgroup's tile, threads.
GEMM_TILES = {0: (128, 128, 512), 1: (64, 64, 256), 2: (32, 32, 256), 3: (16, 16, 512),
              4: (64, 16, 256), 5: (128, 128, 256), 6: (128, 1 << 30, 512), 7: (128, 32, 256),
              8: (128, 64, 256)}


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
    """2^30 rows and a few: only four-wave tiles of 128 rows still fit."""
    assert gemm_route(2 ** 30 + 77, 1, 1) in (5, 7, 8)


# Microseconds on MI355X per kernel (GemmRoute), HIP-graph replays, aligned operands.
GEMM_TIMES = {
    (200, 128, 256): {0: 6.7, 1: 5.0, 2: 3.7, 3: 3.5, 4: 4.7, 6: 6.9, 7: 5.7, 8: 6.3},
    (11264, 96, 288): {0: 10.6, 1: 9.4, 2: 12.4, 3: 37.8, 4: 22.4, 6: 8.4, 7: 9.0, 8: 8.6},
    (4224, 384, 1536): {0: 21.2, 1: 26.0, 2: 41.4, 3: 167.4, 4: 135.7, 7: 30.6, 8: 23.8},
    (40190, 142, 1): {0: 24.8, 1: 18.6, 2: 25.7, 3: 12.9, 4: 12.9, 7: 16.2, 8: 17.2},
    (2865, 337, 277): {0: 29.1, 1: 17.3, 2: 41.0, 3: 45.6, 4: 54.9, 7: 23.3, 8: 24.6},
    (16753, 79, 79): {0: 13.5, 1: 15.9, 2: 20.3, 3: 23.1, 4: 19.6, 7: 14.0, 8: 16.8},
    (17406, 14, 13): {0: 7.4, 1: 5.9, 2: 6.3, 3: 6.1, 4: 3.9, 7: 4.6, 8: 5.5},
    (26803, 2, 9): {0: 6.8, 1: 5.3, 2: 5.5, 3: 7.8, 4: 3.8, 7: 4.4, 8: 5.3},
    (4988, 8, 180): {0: 6.1, 1: 4.7, 2: 5.3, 3: 10.7, 4: 4.5, 6: 4.3, 7: 4.6, 8: 4.8},
    (8030, 20, 168): {0: 6.5, 1: 5.3, 2: 7.0, 3: 14.7, 4: 5.3, 6: 4.4, 7: 5.1, 8: 5.1},
    (60714, 64, 12): {0: 7.5, 1: 6.1, 2: 7.5, 3: 11.7, 4: 6.3, 7: 5.3, 8: 6.0},
    (82454, 4, 56): {0: 12.3, 1: 9.8, 2: 17.3, 3: 46.6, 4: 12.3, 7: 9.2, 8: 8.5},
    (300, 1024, 1024): {0: 22.8, 1: 18.3, 2: 12.0, 3: 22.2, 4: 31.3, 7: 25.0, 8: 26.7},
    (16896, 192, 768): {0: 25.3, 1: 26.1, 2: 51.4, 3: 197.1, 4: 138.8, 7: 29.7, 8: 25.0},
}


@pytest.mark.parametrize("shape", sorted(GEMM_TIMES))
def test_gemm_choice_is_near_the_fastest(shape):
    times = GEMM_TIMES[shape]
    assert times[gemm_route(*shape)] <= 1.1 * min(times.values())


def test_voxel_insertion_launches():
    """One launch where it is faster (24 000 points 48 us, as two 52), two where
    they are (32 000 points 52 us, as one 56)."""
    f = bfhip.hip_lib().bfhip_voxel_insert_launches
    f.argtypes = [C.c_uint]
    assert [f(n) for n in (0, 1000, 17000, 24000, 32000, 100000)] == [1, 1, 1, 1, 2, 2]


def conv_route(d, aligned=True):
    """(ConvRoute + 8 if weights go as float4 + 16 if the patch does, threads)."""
    f = bfhip.hip_lib().bfhip_conv_route
    f.argtypes = [C.c_void_p] * 4 + [C.c_void_p]
    p, threads = 4096 if aligned else 4100, C.c_ulonglong()
    return f(C.byref(d), p, p, p, C.byref(threads)), threads.value


@pytest.mark.parametrize("ci,co", [(1, 1), (1, 33), (3, 64), (8, 8), (8, 129), (64, 1024)])
def test_conv_grids_fit_a_launch(ci, co):
    """Batches of images up to the 2^31 - 1 output pixels a call may have, 1x1,
    3x3, strided and transposed."""
    for h, w in ((1, 1), (7, 5), (64, 64), (1024, 1024), (16000, 16000)):
        for k, s, tr in ((1, 1, 0), (3, 1, 0), (1, 2, 0), (2, 2, 1)):
            oh, ow = (h * s, w * s) if tr else ((h - 1) // s + 1, (w - 1) // s + 1)
            for pixels in (10 ** 5, 2 ** 28, 2 ** 29 + 1, 2 ** 30, 2 ** 30 + 2 ** 28, 2 ** 31 - 1):
                n = max(1, pixels // (oh * ow))
                if n * oh * ow > 2 ** 31 - 1:
                    continue
                d = bfhip.ConvDesc(n, ci, co, h, w, k, k, s, s, 0 if tr else k // 2,
                                   0 if tr else k // 2, oh, ow, tr, 0)
                for aligned in (True, False):
                    assert conv_route(d, aligned)[1] <= LIMIT, (n, h, w, k, s, tr)


def test_conv_route_of_very_many_pixels():
    """1.25 * 2^30 one-channel pixels: more than any direct tile's launch holds
    (4 to 16 threads a pixel), so the gather core's (2) runs."""
    d = bfhip.ConvDesc(20, 1, 1, 8192, 8192, 1, 1, 1, 1, 0, 0, 8192, 8192, 0, 0)
    assert conv_route(d)[0] == 4


def test_conv_planning_is_cheap():
    """Host time of asking for the plans of 200 different 3x3 layers (more than a
    thread keeps) beyond that of layers that are not planned (49 taps), the least
    of 30 runs; planning every tile in full took 2.6 us a layer here."""
    import time
    f = bfhip.hip_lib().bfhip_conv_route
    f.argtypes = [C.c_void_p] * 4 + [C.c_void_p]
    threads = C.c_ulonglong()

    def least(k):
        layers = [bfhip.ConvDesc(6, 256, 256, h, 88, k, k, 1, 1, k // 2, k // 2, h, 88, 0, 0)
                  for h in range(16, 216)]
        args = [(C.addressof(d), 4096, 4096, 4096, C.addressof(threads)) for d in layers]
        best = float("inf")
        for _ in range(30):
            t = time.perf_counter()
            for a in args:
                f(*a)
            best = min(best, time.perf_counter() - t)
        return best / len(layers) * 1e6

    assert least(3) - least(7) < 1.2


def test_conv_plans_kept_by_a_thread():
    """Many layers in turn, each with and without aligned operands, get the plan
    that a thread with nothing kept gives them."""
    import random
    import threading
    rng = random.Random(7)
    calls = []
    for _ in range(60):
        tr = rng.random() < 0.3
        k = 2 if tr else rng.choice((1, 3, 5))
        d = conv_layer(rng.randint(1, 6), rng.randint(1, 200), rng.randint(1, 200), rng.randint(5, 90),
                       rng.randint(5, 120), k, 2 if tr else rng.choice((1, 2)), int(tr))
        calls += [(d, True), (d, False)]
    turn = [rng.choice(calls) for _ in range(600)]
    got = [conv_route(*c) for c in turn]
    fresh = {}
    for i, c in enumerate(calls):
        t = threading.Thread(target=lambda: fresh.__setitem__(i, conv_route(*c)))
        t.start()
        t.join()
    assert got == [fresh[calls.index(c)] for c in turn]


def conv_layer(n, ci, co, h, w, k, s, transpose=0):
    p = 0 if transpose else k // 2
    oh, ow = (h * s, w * s) if transpose else ((h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1)
    return bfhip.ConvDesc(n, ci, co, h, w, k, k, s, s, p, p, oh, ow, transpose, 0)


# Microseconds on MI355X per kernel: the direct tiles with float4 weights (8-11),
# with single floats (0-3), the gather core (4); HIP-graph replays.
CONV_TIMES = {
    (5, 4, 1, 72, 657, 1, 1): {8: 38.3, 9: 30.0, 10: 30.8, 11: 54.3, 0: 40.6, 1: 32.2, 2: 32.7, 3: 58.7, 4: 11.6},
    (5, 8, 8, 187, 470, 1, 1): {8: 82.3, 9: 56.6, 10: 60.4, 11: 110.9, 0: 62.1, 1: 40.0, 2: 44.4, 3: 80.6, 4: 23.5},
    (6, 1, 2, 72, 370, 3, 1): {0: 33.8, 1: 29.1, 2: 26.5, 3: 47.3, 4: 10.2},
    (4, 1, 21, 108, 260, 5, 1): {0: 39.7, 1: 29.1, 2: 28.9, 3: 44.1, 4: 13.4},
    (3, 1, 266, 78, 399, 5, 2): {0: 34.6, 1: 31.7, 2: 47.8, 3: 78.9, 4: 18.7},
    (4, 8, 112, 197, 39, 3, 1): {8: 20.6, 9: 25.4, 10: 32.3, 11: 52.1, 0: 16.0, 1: 17.8, 2: 21.1, 3: 32.8, 4: 26.6},
    (1, 8, 392, 187, 100, 3, 1): {8: 36.9, 9: 37.5, 10: 55.9, 11: 92.9, 0: 27.1, 1: 25.3, 2: 37.0, 3: 58.9, 4: 28.6},
    (2, 88, 16, 110, 411, 1, 1): {8: 28.9, 9: 21.4, 10: 21.5, 11: 35.4, 0: 23.6, 1: 21.2, 2: 15.6, 3: 25.0, 4: 28.3},
    (3, 411, 18, 17, 353, 3, 1): {0: 57.2, 1: 46.5, 2: 33.8, 3: 50.5, 4: 575.1},
    (5, 8, 8, 29, 54, 3, 1): {8: 12.3, 9: 10.3, 10: 7.8, 11: 9.7, 0: 8.4, 1: 7.5, 2: 5.7, 3: 6.6, 4: 14.6},
    (3, 56, 8, 43, 503, 2, 2, 1): {8: 21.4, 9: 16.2, 10: 12.2, 11: 17.1, 1: 19.5, 2: 12.2, 3: 17.7, 4: 151.9},
}


@pytest.mark.parametrize("layer", sorted(CONV_TIMES))
def test_conv_choice_is_near_the_fastest(layer):
    times = CONV_TIMES[layer]
    assert times[conv_route(conv_layer(*layer))[0] % 16] <= 1.1 * min(times.values())
