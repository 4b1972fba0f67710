"""The split-K plan the library reports (ic_gemm_splitk_bytes) for the small-M
shapes of the Flux text stream and the split-K tests, on a 256-CU device
(MI355X; the count the library assumes without a GPU).  Grouped launches pay
for the kernel that adds the slices, so the 512 x 3072 x 3072 grouped W4A8 runs
unsplit (its outputs are then the single fold chain's); the long-K grouped
shapes and the per-row ones keep splitting.  CPU only: the plan is host logic."""
from __future__ import annotations

import pytest


@pytest.mark.parametrize("M,N,K,G,int4,split", [
    (512, 3072, 3072, 24, 1, False),    # Flux text-stream proj, grouped: unsplit
    (512, 3072, 12288, 96, 1, True),    # Flux text-stream MLP-down, grouped
    (256, 3072, 3072, 24, 1, True),     # grouped, fewer tiles
    (64, 3072, 12288, 96, 1, True),     # the split-K tests' shapes
    (100, 1000, 3072, 24, 1, True),
    (512, 3072, 3072, 1, 0, True),      # W8A8 at the text-stream proj shape
    (512, 3072, 3072, 1, 1, True),      # per-row INT4
    (512, 9216, 3072, 24, 1, False),    # enough tiles: no split
    (4608, 3072, 12288, 96, 1, False),  # C3
    (16, 3072, 3072, 24, 1, False),     # the GEMV's rows
])
def test_splitk_plan(rt, M, N, K, G, int4, split):
    nb = rt.lib().ic_gemm_splitk_bytes(M, N, K, G, int4)
    assert (nb > 0) == split, nb
    if split:
        assert nb % (4 * M * N) == 0 and 2 <= nb // (4 * M * N) <= 16


def _shapes():
    return [(M, N, K) for M in (17, 64, 77, 128, 200, 232, 300, 366, 512, 1024)
            for N, K in ((3072, 3072), (5920, 7424), (3856, 7040), (3072, 12288), (1024, 1024))]


def test_no_launch_uses_more_than_the_stated_workspace(rt):
    """ic_gemm_splitk_bytes (ic_gemm_w4a16_splitk_bytes) is the most workspace
    a launch uses: a larger one does not raise the number of slices."""
    for M, N, K in _shapes():
        for weights, G in ((0, 1), (1, 1), (1, K // 128), (0, K // 128), (2, K // 128)):
            stated = (rt.lib().ic_gemm_w4a16_splitk_bytes(M, N, K, G) if weights == 2 else
                      rt.lib().ic_gemm_splitk_bytes(M, N, K, G, weights))
            route = rt.gemm_route(weights, M, N, K, G, workspace_bytes=64 * M * N * 4)
            assert route[3] <= max(1, stated // (4 * M * N)), (weights, M, N, K, G, route)


def test_route_argument_validation(rt):
    for bad in ((3, 1, 1, 1, 1), (0, 0, 8, 128, 1), (0, 8, 8, 128, 3), (1, 1 << 20, 1 << 20, 128, 1)):
        with pytest.raises(RuntimeError):
            rt.gemm_route(*bad, workspace_bytes=0)


@pytest.mark.parametrize("weights", [0, 1, 2])
def test_small_tiles_without_a_workspace(rt, weights):
    """Launches of few tiles take the small ones, unsplit, also where there is no
    workspace (or the shape's plan asks for none)."""
    for M, N, K in ((64, 1024, 1024), (200, 1024, 1024), (256, 4096, 1152)):
        kind, _, _, S = rt.gemm_route(weights, M, N, K, 1, workspace_bytes=0)
        assert (kind, S) == ("small", 1), (M, N, K)


@pytest.mark.parametrize("weights,M,N,K,G,us", [
    # (large, small): measured on MI355X, the launch the small tiles lose to
    (2, 768, 18432, 3072, 24, (89.8, 140)),    # one round of 256 x 256 tiles
    (2, 2048, 7688, 2560, 20, (82.3, 121)),
    (2, 512, 9216, 3072, 24, (64.9, 81)),      # 128 x 64 tiles in two turns per CU
    (2, 384, 12288, 3072, 24, (64.5, 81)),
    (2, 1536, 3072, 3072, 24, (63.7, 79.5)),
    (0, 2048, 12288, 3072, 1, (72.6, 82.2)),
    (0, 2500, 4096, 1152, 1, (20.5, 23.6)),    # short K: the turns' ends weigh
    (1, 640, 12288, 3072, 24, (42.9, 48.1)),
    (1, 384, 18432, 3072, 24, (42.8, 47.6)),
    (1, 4608, 5120, 512, 1, (25.1, 34.6)),     # turns of few stages: their ends weigh
    (1, 1845, 12288, 512, 1, (27.6, 37.9)),
    (1, 4096, 5120, 1024, 1, (33.3, 43.4)),
    (1, 513, 18432, 512, 8, (18.1, 24.0)),     # groups of 64
    (1, 3072, 3904, 256, 8, (18.8, 25.1)),     # groups of 32
    (1, 4608, 5120, 256, 2, (23.5, 29.8)),
])
def test_large_tiles_kept_where_they_lead(rt, weights, M, N, K, G, us):
    assert rt.gemm_route(weights, M, N, K, G)[0] in ("big", "tiles"), us


def test_unpacked_groups_not_on_the_slower_small_tile(rt):
    """384 x 18432 x 3072, int8 weights in groups: 64 x 64 tiles 57 us, 128 x 64
    45.6 and 256 x 192 46.8, which are level."""
    assert rt.gemm_route(0, 384, 18432, 3072, 24)[1:3] in ((128, 64), (256, 192))


@pytest.mark.parametrize("weights,M,N,K,G", [
    (0, 77, 4096, 4096, 1), (0, 512, 3072, 3072, 1), (1, 64, 9216, 3072, 24), (1, 146, 1312, 8448, 132),
    (1, 1357, 2560, 7680, 120), (2, 63, 3256, 3712, 29), (2, 292, 2496, 13312, 104), (0, 512, 3072, 3072, 24),
])
def test_small_tiles_kept_where_they_lead(rt, weights, M, N, K, G):
    assert rt.gemm_route(weights, M, N, K, G)[0] == "small"
