"""The persistent prep kernels with more rows than resident workgroups, so that
every workgroup walks several (alternating row buffers, the next row's DMA behind
this row's stores, no barrier at the top of a row): one to sixteen thousand values,
with and without quantization, against the one-workgroup-per-row kernel (which an
unaligned output row stride selects); the normalising kernels against the oracle
at the first, last and wrapping rows."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {torch.float16: 0, torch.bfloat16: 1}


def _rows_for(dev, width):
    """More than twice the rows that are resident at once: at most 16 waves of
    1024 values per CU."""
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    return cus * max(1, 16 // width) * 2 + 77, cus


def _x(M, K, dtype, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=dev)
    x[:, ::61] *= 20.0
    x *= torch.rand(M, 1, generator=g, device=dev) * 4 + 0.1  # each row its own scale
    return x.to(dtype)


def _prep(rt, K_in, K_w, dtype, dev, use_sr, use_perm):
    g = torch.Generator(device=dev).manual_seed(K_w)
    f = torch.exp(torch.randn(K_in, generator=g, device=dev) * 0.5) if use_sr else None
    p = torch.randperm(K_w, generator=g, device=dev) if use_perm else None
    return f, p, dict(smoothrot=rt.prepare_factors(f, dtype), perm=rt.prepare_perm(p, K_w))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R", [0, 16, 64, 256, 1024, 4096])
@pytest.mark.parametrize("use_sr,use_perm", [(False, False), (True, False), (False, True), (True, True)])
def test_many_rows_equal_the_general_kernel(rt, dev, dtype, R, use_sr, use_perm):
    for w in (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16):
        K_in = 1024 * w - (16 if w % 2 else 0)
        K_w = -(-K_in // max(R, 16)) * max(R, 16)
        M, _ = _rows_for(dev, w)
        x = _x(M, K_in, dtype, dev, w)
        _, _, kw = _prep(rt, K_in, K_w, dtype, dev, use_sr, use_perm)
        kw.update(rot_size=R, w_in=K_w)
        q, s = rt.rotate_quantize(x, **kw)
        q0, s0 = rt.rotate_quantize(x, x_int8_out=torch.empty(M, K_w + 8, dtype=torch.int8, device=dev)[:, :K_w], **kw)
        assert torch.equal(s, s0) and torch.equal(q, q0), (w, K_w)
        y = rt.prepare_activation(x, **kw)
        y0 = rt.prepare_activation(x, out=torch.empty(M, K_w + 4, dtype=dtype, device=dev)[:, :K_w], **kw)
        assert torch.equal(y.view(torch.int16), y0.contiguous().view(torch.int16)), (w, K_w)


@pytest.mark.parametrize("K_in,K_w", [(8208, 8208), (12288, 12288), (12288, 12304), (16384, 16384)])
@pytest.mark.parametrize("use_sr,use_perm", [(True, False), (False, True), (True, True)])
def test_unrotated_rows_at_the_width_rules_line(rt, dev, K_in, K_w, use_sr, use_perm):
    """bf16: wide tiles up to six rows per CU, three or four tiles of four waves
    beyond."""
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    for M in (6 * cus, 6 * cus + 1):
        x = _x(M, K_in, torch.bfloat16, dev, M)
        _, _, kw = _prep(rt, K_in, K_w, torch.bfloat16, dev, use_sr, use_perm)
        q, s = rt.rotate_quantize(x, w_in=K_w, **kw)
        q0, s0 = rt.rotate_quantize(x, w_in=K_w, x_int8_out=torch.empty(M, K_w + 8, dtype=torch.int8, device=dev)[:, :K_w],
                                    **kw)
        assert torch.equal(s, s0) and torch.equal(q, q0), M


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R", [64, 256])
@pytest.mark.parametrize("use_sr,use_perm", [(False, False), (True, False), (False, True), (True, True)])
def test_five_thousand_values_at_the_width_rules_line(rt, dev, dtype, R, use_sr, use_perm):
    """One wide tile up to three rows per CU, two narrow ones beyond."""
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    for K_in in (4112, 5120):
        K_w = -(-K_in // R) * R
        for M in (3 * cus, 3 * cus + 1, 7 * cus + 1):
            x = _x(M, K_in, dtype, dev, M)
            _, _, kw = _prep(rt, K_in, K_w, dtype, dev, use_sr, use_perm)
            q, s = rt.rotate_quantize(x, rot_size=R, w_in=K_w, **kw)
            q0, s0 = rt.rotate_quantize(x, rot_size=R, w_in=K_w,
                                        x_int8_out=torch.empty(M, K_w + 8, dtype=torch.int8, device=dev)[:, :K_w], **kw)
            assert torch.equal(s, s0) and torch.equal(q, q0), (M, K_in)


def _norm_rows_match(rt, oracle, dev, x, rows, R, K_w, dtype, norm, use_sr, use_perm):
    K_in = x.shape[1]
    f, p, kw = _prep(rt, K_in, K_w, dtype, dev, use_sr, use_perm)
    g = torch.Generator(device=dev).manual_seed(1)
    nw = 1 + 0.2 * torch.randn(K_in, generator=g, device=dev)
    nb = 0.1 * torch.randn(K_in, generator=g, device=dev)
    q, s = rt.norm_rotate_quantize(x, norm=norm, weight=nw, bias=nb, eps=1e-6, rot_size=R, w_in=K_w, **kw)
    rq, rs = oracle.norm_rotate_quantize(
        x[rows].cpu(), DT[dtype], norm, nw.cpu().numpy(), nb.cpu().numpy(), 1e-6,
        smoothrot=f.cpu().numpy() if use_sr else None, rot_size=R, w_in=K_w, perm=p.cpu().numpy() if use_perm else None)
    assert np.array_equal(s[rows].cpu().numpy(), rs), (R, K_w, x.shape[0])
    assert np.array_equal(q[rows].cpu().numpy(), rq), (R, K_w, x.shape[0])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("norm", ["layer", "rms"])
@pytest.mark.parametrize("use_sr,use_perm", [(False, False), (True, False), (False, True), (True, True)])
def test_normalised_rows_at_the_width_rules_lines(rt, oracle, dev, dtype, norm, use_sr, use_perm):
    """R = 1024, five or six thousand values: one wide tile up to a row per CU,
    two narrow ones beyond, under two register bounds; R = 4096, one tile: two
    bounds as well."""
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    for K_in, K_w in ((4112, 5120), (5120, 5120), (5136, 6144), (6144, 6144)):
        for M in (1, cus, cus + 1, 2 * cus + 1, 4 * cus, 4 * cus + 1):
            x = _x(M, K_in, dtype, dev, M)
            _norm_rows_match(rt, oracle, dev, x, sorted({0, M // 2, M - 1}), 1024, K_w, dtype, norm, use_sr, use_perm)
    for K_in in (1040, 4096):
        for M in (1, 2 * cus, 2 * cus + 1, 4 * cus, 4 * cus + 1):
            x = _x(M, K_in, dtype, dev, M)
            _norm_rows_match(rt, oracle, dev, x, sorted({0, M // 2, M - 1}), 4096, 4096, dtype, norm, use_sr, use_perm)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("norm", ["layer", "rms"])
@pytest.mark.parametrize("use_sr,use_perm", [(False, False), (True, False), (False, True), (True, True)])
def test_many_normalised_rows_match_oracle(rt, oracle, dev, dtype, norm, use_sr, use_perm):
    for R, w in ((16, 1), (256, 2), (64, 3), (0, 4), (256, 5), (1024, 5), (0, 6), (1024, 6), (64, 7), (256, 8), (0, 11),
                 (256, 12), (1024, 14), (4096, 16)):
        K_in = 1024 * w - (16 if w % 2 else 0)
        K_w = -(-K_in // max(R, 16)) * max(R, 16)
        M, cus = _rows_for(dev, w)
        x = _x(M, K_in, dtype, dev, w + R)
        rows = sorted({0, M // 2, M - 1} | {cus * n + d for n in (1, 2, 4) for d in (0, 1) if cus * n + d < M})
        _norm_rows_match(rt, oracle, dev, x, rows, R, K_w, dtype, norm, use_sr, use_perm)
