"""The small-tile GEMM kernel on 17 to a few hundred tokens: the shapes below
take its 32 x 64 tile (a few 64 x 64), from one K stage to many and in K slices,
with groups of one to several stages; test_gpu_gemm_tiles.py has every tile.

INT8 modes: bit-equal to the scalar kernel (unaligned operand rows select it),
which folds the same blocks in the same order; per-row K splits are exact
int32 sums, so they are bit-equal too.  W4A16: within the fp32 summation bound
of the float64 product of the dequantized weights, K 2^-24 sum |x w| (any
order of K fp32 additions), plus the output's rounding."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(17, 8, 128), (32, 64, 384), (33, 72, 1152), (64, 200, 512), (65, 64, 2560), (129, 136, 640),
          (200, 1000, 1024), (300, 264, 3072)]


def _unaligned(x):
    """The same rows on a row stride that is not a multiple of 16 bytes."""
    wide = torch.zeros(x.shape[0], x.shape[1] + 3, dtype=x.dtype, device=x.device)
    wide[:, : x.shape[1]] = x
    return wide[:, : x.shape[1]]


def _codes(M, K, g, dev):
    x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    x[0] = 127  # the largest sums
    return x.to(dev)


@pytest.mark.parametrize("mode", ["row8", "row4", "g128", "g64", "g32", "g96", "unpacked", "unpacked256"])
@pytest.mark.parametrize("epi", [False, True])
def test_int8_modes_equal_the_scalar_kernel(rt, dev, mode, epi):
    for M, N, K in SHAPES:
        gs = {"row8": K, "row4": K, "g128": 128, "g64": 64, "g32": 32, "g96": 96, "unpacked": 128,
              "unpacked256": 256}[mode]
        if K % gs:
            K = -(-K // (gs * 128)) * gs * 128
            gs = K if mode in ("row8", "row4") else gs
        g = torch.Generator().manual_seed(M * 7 + K)
        dt = torch.float16 if M % 2 else torch.bfloat16
        x = _codes(M, K, g, dev)
        s_a = (torch.rand(M, generator=g) * 1e-2).to(dev)
        s_w = (torch.rand(N, K // gs, generator=g) * 1e-2).to(dev)
        kw = dict(bias=torch.randn(N, generator=g).to(dt).to(dev), out_dtype=dt)
        if epi:
            kw.update(activation=3, residual=torch.randn(M, N, generator=g).to(dt).to(dev))
        if mode == "row8":
            w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(dev)
            ref = rt.fused_int8_gemm_dequant(_unaligned(x), w, s_w, s_a, **kw)
            assert torch.equal(rt.fused_int8_gemm_dequant(x, w, s_w, s_a, **kw), ref), (M, N, K)
            continue
        w = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8).to(dev)
        ref = rt.gemm_w4a8(_unaligned(x), w, s_w, s_a, **kw)
        split = gs % 128 == 0 and K // gs > 1 and rt.lib().ic_gemm_splitk_bytes(M, N, K, K // gs, 1) > 0
        if mode.startswith("unpacked"):
            outs = [rt.gemm_w4a8_unpacked(x, rt.unpack_int4_to_int8(w, K), s_w, s_a, **kw)]
        else:
            outs = [rt.gemm_w4a8(x, w, s_w, s_a, **kw),
                    rt.gemm_w4a8(x, rt.int4_interleave_k(w), s_w, s_a, kil=True, **kw)]
        for out in outs:
            if split:  # the slices of a grouped fold are added in slice order
                d = (out.float() - ref.float()).abs()
                assert float((d / ref.float().abs().clamp_min(1.0)).max()) < 2 ** -6
            else:
                assert torch.equal(out, ref), (M, N, K)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("group", [64, 128, 0])
def test_w4a16_small_tiles(rt, dev, dtype, group):
    for M, N, K in SHAPES + [(31, 96, 9216), (140, 72, 4096)]:
        g = torch.Generator().manual_seed(M + K)
        gs = group or K
        x = torch.randn(M, K, generator=g).to(dtype).to(dev)
        w = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8).to(dev)
        s = (torch.rand(N, K // gs, generator=g) * 1e-2 + 1e-3).to(dev)
        b = torch.randn(N, generator=g).to(dtype).to(dev)
        wf = rt.unpack_int4_to_float(w, s, K, dtype).double()
        ref = x.double() @ wf.t().contiguous() + b.double()
        ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
        bound = (K + 16) * 2.0 ** -24 * (x.double().abs() @ wf.abs().t().contiguous()) + ulp * ref.abs() * 1.01 + 1e-6
        out = rt.gemm_w4a16(x, w, s, bias=b)
        assert bool(((out.double() - ref).abs() <= bound).all()), (M, N, K)
        assert torch.equal(out, rt.gemm_w4a16(x, w, s, bias=b))
        if rt.w4a16_staged_pays(M, N, K, K // gs):
            assert torch.equal(rt.gemm_w4a16_staged(x, *rt.w4a16_stage_layout(w, s), bias=b), out)
        # without a workspace: unsplit
        o2 = torch.empty_like(out)
        rt._call("ic_gemm_w4a16", rt._ptr(x), rt._dt(dtype, ""), M, K, K, rt._ptr(w), N, K // 2, rt._ptr(s), K // gs,
                 rt._ptr(b), rt._dt(dtype, ""), rt._ptr(o2), N, rt._stream(x))
        assert bool(((o2.double() - ref).abs() <= bound).all()), (M, N, K)


def test_workspace_not_aligned_to_16_bytes(rt, dev):
    """The split reductions load 16 bytes of partials at a time; any workspace
    that was accepted before still is, and gives the same results."""
    M, N, K = 40, 256, 8192
    g = torch.Generator().manual_seed(5)
    st, bf = rt._stream(torch.empty(1, device=dev)), rt._dt(torch.bfloat16, "")
    x, s_a = _codes(M, K, g, dev), (torch.rand(M, generator=g) * 1e-2).to(dev)
    xf = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
    w8 = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(dev)
    w4 = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8).to(dev)
    s_w = (torch.rand(N, K // 128, generator=g) * 1e-2).to(dev)
    s_row = s_w[:, 0].contiguous()
    size = max(rt.lib().ic_gemm_splitk_bytes(M, N, K, G, i4) for G, i4 in ((1, 0), (K // 128, 1)))
    size = max(size, rt.lib().ic_gemm_w4a16_splitk_bytes(M, N, K, K // 128))
    assert size > 0
    buf = torch.empty(size + 64, dtype=torch.uint8, device=dev)
    p = rt._ptr

    def run(entry, *args, ws):
        out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        tail = (p(buf[ws:]), size) if ws is not None else ()
        rt._call(entry, *args[:-1], *args[-1], p(out), *((bf,) if "w4a16" not in entry else ()), N, *tail, st)
        return out

    a8 = (p(x), M, K, K, p(w8), N, K, p(s_a), p(s_row), (None, 0))
    a4 = (p(x), M, K, K, p(w4), N, K // 2, p(s_w), K // 128, p(s_a), (None, 0))
    a16 = (p(xf), bf, M, K, K, p(w4), N, K // 2, p(s_w), K // 128, (None, 0))
    for ws in (4, 8):
        assert torch.equal(run("ic_gemm_w8a8_ws", *a8, ws=ws), run("ic_gemm_w8a8_ws", *a8, ws=0))
        assert torch.equal(run("ic_gemm_w4a8_ws", *a4, ws=ws), run("ic_gemm_w4a8_ws", *a4, ws=0))
        assert torch.equal(run("ic_gemm_w4a16_ws", *a16, ws=ws), run("ic_gemm_w4a16", *a16, ws=None))
