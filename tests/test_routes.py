"""Which kernel sq_linear_gemm takes, as its host functions plan it (for 256 compute units where there is no GPU; no pointer is followed)."""

import ctypes
import math
import random

from quantexperiments_amd import _lib

FUSED, COLUMNS, MID, PASSES, DECODED, TILES, TILES_IN_PLANE_ORDER = range(1, 8)


def _stack(rows, C, d, bits, G=1):
    pieces, off = [], 0
    for R in rows:
        m = _lib.SqMatrix()
        m.tags = m.table = m.row_scale = 4096
        m.row_book = 4096 if G > 1 else None
        m.stream = 4096 if d == 4 else None
        m.R, m.C, m.d, m.bits, m.G, m.M, m.W, m.y_off = R, C, d, bits, G, 1, (C // d * bits + 31) // 32, off
        off += R
        pieces.append(m)
    return _lib.matrix_array(pieces)


def _kernel(rows, C, d, bits, G, T, dtype=_lib.SQ_BF16):
    us = (ctypes.c_float * 3)()
    return _lib.lib().sq_gemm_kernel_for_tests(_stack(rows, C, d, bits, G), len(rows), T, dtype, us), list(us)


def _log(rng, lo, hi):
    return round(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def _rows(rng):
    first = _log(rng, 256, 19000)
    return rng.choice(([first], [first, first], [first, max(64, first // 4), max(64, first // 4)]))


def test_a_kernel_is_given_up_for_the_one_it_was_compared_with():
    """d = 4 at 129 to 768 rows: what the fused kernel has a cut for runs there, or on the kernel of small products where that is estimated to take 85 % of its
    time, also beyond the row counts that always run there, or in tiles where those are not estimated to take more than 1 / 0.73 of that again."""
    rng = random.Random(5)
    seen = set()
    for _ in range(6000):
        rows, C, bits, T = _rows(rng), max(512, _log(rng, 512, 9000) // 64 * 64), rng.choice((8, 10, 12)), rng.randint(129, 768)
        G = rng.choice((1, 1, 1, 4))
        k, us = _kernel(rows, C, 4, bits, G, T)
        if us[0] > 1e29:
            continue
        seen.add(k)
        if k == FUSED:
            assert us[1] > 80 or us[1] > 0.849 * us[0], (rows, C, bits, G, T, us)
        else:
            assert us[1] < 0.851 * us[0] and (k == MID or (k == TILES and us[2] < us[1] / 0.729)), (rows, C, bits, G, T, us)
    assert seen == {FUSED, MID, TILES}
    for case in (([7704], 8192, 4, 10, 4, 262), ([9792, 9792], 3200, 4, 12, 1, 260), ([6987, 1746, 1746], 4800, 4, 12, 1, 429), ([10752, 10752], 2880, 4, 8, 1, 325)):
        assert _kernel(*case)[0] == MID


def test_two_blocks_of_tokens_are_compared_with_the_tiles():
    """d = 8 at 385 to 768 rows: the fused kernel's one round of two blocks of tokens gives way to a decode and tiles where those are estimated to take less, whatever type x has
    and whichever order their decode takes, and the kernel of small products is compared with the tiles of x's own type."""
    for dtype in (_lib.SQ_BF16, _lib.SQ_F16):
        assert _kernel([18944], 3584, 8, 16, 1, 450, dtype)[0] == TILES_IN_PLANE_ORDER
        for case in (([9394, 9394], 576, 498), ([7749, 1937, 1937], 448, 483), ([10009, 10009], 13568, 490)):
            assert _kernel(case[0], case[1], 8, 16, 1, case[2], dtype)[0] == FUSED
    rng = random.Random(6)
    seen, types = set(), 0
    for _ in range(4000):
        rows, C, T, dtype = _rows(rng), max(192, _log(rng, 192, 14000) // 64 * 64), rng.randint(385, 768), rng.choice((_lib.SQ_BF16, _lib.SQ_F16))
        k, us = _kernel(rows, C, 8, 16, 1, T, dtype)
        if us[0] < 1e29:
            seen.add((k, dtype))
            assert (k == FUSED) == (us[2] >= us[0]), (rows, C, T, us)
        elif k in (MID, TILES, TILES_IN_PLANE_ORDER):
            types += _kernel(rows, C, 8, 16, 1, T, _lib.SQ_BF16)[1][2] != _kernel(rows, C, 8, 16, 1, T, _lib.SQ_F16)[1][2]
            assert (k == MID) == (us[1] < (0.9 if us[1] < 50 else 0) * us[2]), (rows, C, T, us)
    assert seen >= {(k, t) for k in (FUSED, TILES, TILES_IN_PLANE_ORDER) for t in (_lib.SQ_BF16, _lib.SQ_F16)} and types
