"""Shapes that reach each output tile of the GEMM kernels, found by asking the
library which kernel a shape takes (gemm_route): more than one tile each way and
ragged against it, the smallest of a list of candidates first."""
from __future__ import annotations

import functools

# mode: weights argument of gemm_route, columns per group (0: per row), K stage
MODES = {"row8": (0, 0, 128), "row4": (1, 0, 128), "g128": (1, 128, 128), "g64": (1, 64, 128), "g32": (1, 32, 128),
         "unpacked": (0, 128, 128), "w4a16": (2, 64, 64)}
_SMALL_M = (17, 33, 49, 65, 97, 113, 129, 161, 201, 257, 333, 385, 449, 515, 601, 701, 901, 1025, 1201)
_SMALL_N = (8, 72, 136, 200, 520, 1000, 1544, 2056, 2568, 3080, 4104, 5128, 6152, 7176, 8200, 9224, 10248, 12296)
_BIG_M = (129, 201, 257, 301, 401, 601, 901, 1301, 1801, 2301, 2901, 3501, 4301, 5121)
_BIG_N = (200, 520, 1000, 2056, 3080, 4104, 6152, 8200, 10248, 12296)


def groups(mode: str, K: int) -> int:
    gs = MODES[mode][1]
    return K // gs if gs else 1


def ragged(M: int, N: int, rows: int, cols: int) -> bool:
    return M % rows != 0 and N % cols != 0 and N > cols


@functools.lru_cache(maxsize=None)
def _candidates(big: bool):
    return sorted(((m, n) for m in (_BIG_M if big else _SMALL_M) for n in (_BIG_N if big else _SMALL_N)),
                  key=lambda mn: mn[0] * mn[1])


def find(rt, mode: str, kind: str, rows: int, cols: int, K: int, split: bool | None = None):
    """(M, N, K slices) of the smallest candidate on that kernel and tile, or None."""
    if MODES[mode][1] and groups(mode, K) < 2 and mode not in ("w4a16",):
        return None  # one group is the per-row mode
    one_row = None  # the fallback where only single rows of tiles take it
    for M, N in _candidates(kind == "big"):
        route = rt.gemm_route(MODES[mode][0], M, N, K, groups(mode, K))
        if route[:3] == (kind, rows, cols) and ragged(M, N, rows, cols) and split in (None, route[3] > 1):
            if M > rows:
                return M, N, route[3]
            one_row = one_row or (M, N, route[3])
    return one_row


# tiles each mode has
SMALL_TILES = [(mode, *tile) for mode in MODES for tile in ((32, 64), (64, 64), (128, 64), (128, 128))
               if tile[0] < 128 or mode in ("row8", "w4a16") or (tile == (128, 64) and mode != "row4")]
# a mode's tiles that K is split on by the plan of some candidate
SPLIT_TILES = [("row8", 32, 64), ("row8", 64, 64), ("row8", 128, 64), ("row8", 128, 128), ("row4", 32, 64), ("row4", 64, 64),
               ("g128", 32, 64), ("g128", 64, 64), ("g128", 128, 64), ("unpacked", 32, 64), ("unpacked", 64, 64),
               ("w4a16", 32, 64), ("w4a16", 64, 64), ("w4a16", 128, 64), ("w4a16", 128, 128)]
BIG_TILES = [(mode, rows, 192) for mode in MODES for rows in (256, 288, 320)] + [("w4a16", 256, 256), ("w4a16", 288, 256)]


def small_unsplit(rt, mode, rows, cols):
    """[(M, N, K)]: from one K stage on (the rings have two to four slots)."""
    stage = MODES[mode][2]
    return [(s[0], s[1], n * stage) for n in (1, 2, 3, 4, 5, 6, 9, 12) if (s := find(rt, mode, "small", rows, cols, n * stage, False))]


def small_split(rt, mode, rows, cols):
    for K in (1024, 1536, 2048, 4096, 8192):
        s = find(rt, mode, "small", rows, cols, K, True)
        if s:
            return s[0], s[1], K, s[2]
    return None


def big(rt, mode, rows, cols, stages):
    K = stages * MODES[mode][2]
    s = find(rt, mode, "big", rows, cols, K)
    return s and (s[0], s[1], K)


def tile_kernel(rt, mode, split, odd_columns=0):
    """(M, N, K, slices) of a shape that stays on the tile kernel, in K slices or
    not; odd_columns: added to a multiple of 8 columns, which no other kernel takes."""
    for K in (3072, 8192, 12288) if split else (384, 1024, 3072):
        for M, N in _candidates(True):
            route = rt.gemm_route(MODES[mode][0], M, N + odd_columns, K, groups(mode, K))
            if route[0] == "tiles" and (route[3] > 1) == split and ragged(M, N + odd_columns, route[1], route[2]):
                return M, N + odd_columns, K, route[3]
    return None


# packed INT4 in K slices: the small tiles lead wherever the output is aligned
TILE_KERNEL = [(mode, split, odd) for mode in ("row8", "row4", "g128", "unpacked") for split in (False, True)
               for odd in (0, 1, 4) if (mode, split, odd) not in (("row4", True, 0), ("g128", True, 0))]
