"""The single-pass prep kernels over every workgroup width (one to eight, twelve
waves, two tiles) at its smallest, a ragged and its largest row: codes and scales
equal to the one-workgroup-per-row kernel (a code row stride that is not a
multiple of 16 selects it), and the normalising kernels to the oracle's
composition.  Values include exact rounding midpoints, zeros and subnormals."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {torch.float16: 0, torch.bfloat16: 1}


def _rows(M, K, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    x[:, :: 61] *= 20.0
    x = x.to(dtype)
    x[1] = 0
    x[2] = (torch.randn(K, generator=g) * 1e-6).to(dtype)
    # few significant bits: most rotated sums lie on or next to midpoints
    x[3] = torch.randint(-3, 4, (K,), generator=g).to(dtype) + (torch.randint(0, 2, (K,), generator=g) * 2.0 ** -7).to(dtype)
    return x


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R", [0, 16, 64, 256, 1024])
@pytest.mark.parametrize("use_sr,use_perm", [(False, False), (True, False), (True, True)])
def test_codes_equal_the_general_kernel_at_every_width(rt, dev, dtype, R, use_sr, use_perm):
    for w in (1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 14, 15, 16):
        for K_w in (1024 * (w - 1) + max(R, 16), 1024 * w):
            if R == 1024 and K_w % 1024:
                continue
            K_in = K_w if K_w == 1024 * w else max(16, K_w - 16 * (R > 16))
            M = 5 if w % 2 else 600
            if M == 600 and w > 8:
                M = 40
            g = torch.Generator().manual_seed(K_w)
            x = _rows(M, K_in, dtype, K_w + M).to(dev)
            sr = rt.prepare_factors(torch.exp(torch.randn(K_in, generator=g) * 0.5).to(dev), dtype) if use_sr else None
            pp = rt.prepare_perm(torch.randperm(K_w, generator=g).to(dev), K_w) if use_perm else None
            kw = dict(rot_size=R, w_in=K_w, smoothrot=sr, perm=pp)
            q, s = rt.rotate_quantize(x, **kw)
            q0 = torch.empty(M, K_w + 8, dtype=torch.int8, device=dev)[:, :K_w]
            q0, s0 = rt.rotate_quantize(x, x_int8_out=q0, **kw)
            assert torch.equal(s, s0), (w, K_w)
            assert torch.equal(q, q0), (w, K_w)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("norm", ["layer", "rms"])
@pytest.mark.parametrize("K,K_w,R,prep", [(512, 512, 16, True), (1040, 1088, 64, False), (2560, 2560, 256, True),
                                          (5120, 5120, 256, True), (6144, 6144, 64, False), (5136, 6144, 1024, True),
                                          (6400, 6400, 256, False), (7168, 7168, 0, True), (8192, 8192, 256, True),
                                          (10240, 10240, 256, False), (13312, 14336, 64, True)])
def test_norm_widths_match_oracle(rt, oracle, dev, dtype, norm, K, K_w, R, prep):
    g = torch.Generator().manual_seed(K + R)
    x = (torch.randn(9, K, generator=g) * 2 + 0.3).to(dtype)
    w = 1 + 0.2 * torch.randn(K, generator=g)
    b = 0.1 * torch.randn(K, generator=g)
    sr = torch.exp(torch.randn(K, generator=g) * 0.5) if prep else None
    perm = torch.randperm(K_w, generator=g) if prep else None
    q, s = rt.norm_rotate_quantize(
        x.to(dev), norm=norm, weight=w.to(dev), bias=b.to(dev), eps=1e-6, rot_size=R, w_in=K_w,
        smoothrot=rt.prepare_factors(sr.to(dev), dtype) if prep else None,
        perm=rt.prepare_perm(perm.to(dev), K_w) if prep else None)
    rq, rs = oracle.norm_rotate_quantize(
        x, DT[dtype], norm, w.numpy(), b.numpy(), 1e-6, smoothrot=sr.numpy() if prep else None, rot_size=R, w_in=K_w,
        perm=perm.numpy() if prep else None)
    assert np.array_equal(s.cpu().numpy(), rs)
    assert np.array_equal(q.cpu().numpy(), rq)
