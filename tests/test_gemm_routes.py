"""Every tile of the small- and big-tile GEMM kernels is what the library's plan
chooses for some ragged shape (tests/_tiles.py), so that the GPU tests built on
those shapes cover it whatever the plan's constants are.  CPU only: the plan is
host arithmetic."""
from __future__ import annotations

import pytest

import _tiles


@pytest.mark.parametrize("mode,rows,cols", _tiles.SMALL_TILES)
def test_small_tiles_are_reached(rt, mode, rows, cols):
    shapes = _tiles.small_unsplit(rt, mode, rows, cols)
    assert len(shapes) >= 3, shapes


@pytest.mark.parametrize("mode,rows,cols", _tiles.SPLIT_TILES)
def test_split_tiles_are_reached(rt, mode, rows, cols):
    assert _tiles.small_split(rt, mode, rows, cols)


@pytest.mark.parametrize("mode,rows,cols", _tiles.BIG_TILES)
def test_big_tiles_are_reached(rt, mode, rows, cols):
    assert _tiles.big(rt, mode, rows, cols, 3)
    if mode == "w4a16":
        assert _tiles.big(rt, mode, rows, cols, 129)  # the three-slot ring


@pytest.mark.parametrize("mode,split,odd", _tiles.TILE_KERNEL)
def test_tile_kernel_is_reached(rt, mode, split, odd):
    assert _tiles.tile_kernel(rt, mode, split, odd)


def test_other_kernels(rt):
    assert rt.gemm_route(rt.IC_WEIGHTS_I8, 16, 3072, 3072, 1)[0] == "gemv"
    assert rt.gemm_route(rt.IC_WEIGHTS_W4A16, 2, 9216, 3072, 24)[0] == "gemv"
    assert rt.gemm_route(rt.IC_WEIGHTS_I4, 37, 96, 520, 1)[0] == "scalar"
    assert rt.gemm_route(rt.IC_WEIGHTS_I4, 300, 1001, 1024, 8)[0] == "tiles"  # N not a multiple of 8
    assert rt.gemm_route(rt.IC_WEIGHTS_W4A16, 300, 1024, 1024, 32)[0] == "tiles"  # groups of 32
