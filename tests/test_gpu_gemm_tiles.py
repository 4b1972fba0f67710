"""Each output tile of the small- and big-tile GEMM kernels, and the tile kernel
where it is still chosen, on ragged shapes that the library's plan gives it
(tests/_tiles.py): one K stage to past the ring's depth, K slices, packed (both
nibble orders), unpacked and staged weights, with and without bias, activation and
residual.

INT8 modes: bit-equal to the scalar kernel (unaligned operand rows select it),
which folds the same blocks in the same order; per-row K slices are exact int32
sums.  Grouped slices fold their groups apart and add S partial folds: both
orders are within (G + S) 2^-24 sum |block sum * scale| of the exact fold, so
within twice that of each other, plus one rounding of the output.  W4A16: within
the fp32 summation bound of the float64 product of the dequantized weights, K
2^-24 sum |x w| (any order of K fp32 additions), plus the output's rounding."""
from __future__ import annotations

import pytest
import torch

import _tiles

pytestmark = pytest.mark.gpu
ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _unaligned(x):
    """The same rows on a row stride that is not a multiple of 16 bytes."""
    wide = torch.zeros(x.shape[0], x.shape[1] + 3, dtype=x.dtype, device=x.device)
    wide[:, : x.shape[1]] = x
    return wide[:, : x.shape[1]]


def _int8_operands(mode, M, N, K, dev):
    g = torch.Generator(device=dev).manual_seed(M * 7 + N + K)
    x = torch.randint(-127, 128, (M, K), generator=g, device=dev, dtype=torch.int8)
    x[0] = 127  # the largest sums
    s_a = torch.rand(M, generator=g, device=dev) * 1e-2
    s_w = torch.rand(N, _tiles.groups(mode, K), generator=g, device=dev) * 1e-2
    if mode == "row8":
        w = torch.randint(-127, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    else:
        w = torch.randint(0, 256, (N, K // 2), generator=g, device=dev, dtype=torch.uint8)
    return x, w, s_w, s_a, g


def _int8_outputs(rt, mode, x, w, s_w, s_a, kw):
    """The scalar kernel's output and those of the mode's weight forms."""
    if mode == "row8":
        return rt.fused_int8_gemm_dequant(_unaligned(x), w, s_w, s_a, **kw), [
            rt.fused_int8_gemm_dequant(x, w, s_w, s_a, **kw)]
    ref = rt.gemm_w4a8(_unaligned(x), w, s_w, s_a, **kw)
    if mode == "unpacked":
        return ref, [rt.gemm_w4a8_unpacked(x, rt.unpack_int4_to_int8(w, x.shape[1]), s_w, s_a, **kw)]
    return ref, [rt.gemm_w4a8(x, w, s_w, s_a, **kw), rt.gemm_w4a8(x, rt.int4_interleave_k(w), s_w, s_a, kil=True, **kw)]


def _check_int8(rt, dev, mode, M, N, K, epi, slices=1):
    print(f"[{mode}] {M} x {N} x {K} epi={epi} slices={slices}", flush=True)
    x, w, s_w, s_a, g = _int8_operands(mode, M, N, K, dev)
    dt = torch.float16 if (M + K // 128) % 2 else torch.bfloat16
    kw = dict(out_dtype=dt)
    if epi:
        kw.update(bias=torch.randn(N, generator=g, device=dev).to(dt), activation=3,
                  residual=torch.randn(M, N, generator=g, device=dev).to(dt))
    ref, outs = _int8_outputs(rt, mode, x, w, s_w, s_a, kw)
    for out in outs:
        if slices == 1 or s_w.shape[1] == 1:
            assert torch.equal(out, ref)
            continue
        wq = rt.unpack_int4_to_int8(w, K).double().reshape(N, s_w.shape[1], -1)
        size = x.double().abs() @ (wq * s_w.double().unsqueeze(2)).reshape(N, K).abs().t().contiguous()
        bound = 2 * (s_w.shape[1] + slices) * 2.0 ** -24 * size * s_a.double().unsqueeze(1)
        if epi:
            bound = bound * 1.13  # the largest slope of GELU
        bound = bound + 2 * ULP[dt] * ref.double().abs() + 1e-6
        assert bool(((out.double() - ref.double()).abs() <= bound).all())


def _check_w4a16(rt, dev, M, N, K, group, dtype):
    print(f"[w4a16] {M} x {N} x {K} group={group} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(dtype)
    w = torch.randint(0, 256, (N, K // 2), generator=g, device=dev, dtype=torch.uint8)
    s = torch.rand(N, K // group, generator=g, device=dev) * 1e-2 + 1e-3
    b = torch.randn(N, generator=g, device=dev).to(dtype)
    wt = rt.unpack_int4_to_float(w, s, K, dtype).double().t().contiguous()
    ref = x.double() @ wt + b.double()
    bound = (K + 16) * 2.0 ** -24 * (x.double().abs() @ wt.abs()) + ULP[dtype] * ref.abs() * 1.01 + 1e-6
    del wt
    out = rt.gemm_w4a16(x, w, s, bias=b)
    assert bool(((out.double() - ref).abs() <= bound).all())
    if rt.w4a16_staged_pays(M, N, K, K // group):
        assert torch.equal(rt.gemm_w4a16_staged(x, *rt.w4a16_stage_layout(w, s), bias=b), out)
    else:
        assert M <= 128


@pytest.mark.parametrize("mode,rows,cols", [t for t in _tiles.SMALL_TILES if t[0] != "w4a16"])
@pytest.mark.parametrize("epi", [False, True])
def test_small_tile_int8(rt, dev, mode, rows, cols, epi):
    shapes = _tiles.small_unsplit(rt, mode, rows, cols)
    assert len(shapes) >= 3
    for M, N, K in shapes:
        _check_int8(rt, dev, mode, M, N, K, epi)


@pytest.mark.parametrize("mode,rows,cols", [t for t in _tiles.SPLIT_TILES if t[0] != "w4a16"])
@pytest.mark.parametrize("epi", [False, True])
def test_small_tile_int8_split(rt, dev, mode, rows, cols, epi):
    M, N, K, slices = _tiles.small_split(rt, mode, rows, cols)
    _check_int8(rt, dev, mode, M, N, K, epi, slices)


@pytest.mark.parametrize("rows,cols", [t[1:] for t in _tiles.SMALL_TILES if t[0] == "w4a16"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_small_tile_w4a16(rt, dev, rows, cols, dtype):
    shapes = _tiles.small_unsplit(rt, "w4a16", rows, cols)
    assert len(shapes) >= 3
    for M, N, K in shapes + [_tiles.small_split(rt, "w4a16", rows, cols)[:3]]:
        _check_w4a16(rt, dev, M, N, K, 64, dtype)


@pytest.mark.parametrize("mode,rows,cols", [t for t in _tiles.BIG_TILES if t[0] != "w4a16"])
@pytest.mark.parametrize("epi", [False, True])
def test_big_tile_int8(rt, dev, mode, rows, cols, epi):
    _check_int8(rt, dev, mode, *_tiles.big(rt, mode, rows, cols, 3), epi)


@pytest.mark.parametrize("mode,split,odd", _tiles.TILE_KERNEL)
@pytest.mark.parametrize("epi", [False, True])
def test_tile_kernel_int8(rt, dev, mode, split, odd, epi):
    M, N, K, slices = _tiles.tile_kernel(rt, mode, split, odd)
    _check_int8(rt, dev, mode, M, N, K, epi, slices)


@pytest.mark.parametrize("rows,cols", [t[1:] for t in _tiles.BIG_TILES if t[0] == "w4a16"])
@pytest.mark.parametrize("stages", [3, 129])  # the two- and the three-slot ring
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_big_tile_w4a16(rt, dev, rows, cols, stages, dtype):
    _check_w4a16(rt, dev, *_tiles.big(rt, "w4a16", rows, cols, stages), 64, dtype)
