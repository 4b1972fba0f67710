"""The single-pass preparation kernels without quantization (ic_prepare_activation)
against the one-workgroup-per-row kernel they stand in for, which an output row
stride that is not a multiple of 8 values selects: the same bits over dtypes,
rotations, row widths (every tile count and workgroup width), pads, factors,
perms, row strides, in-place use, and rows of zeros, subnormals, infinities
and NaN."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

WIDTHS = {0: [16, 3072, 8208, 16384], 16: [64, 4096, 6144], 64: [64, 1088, 3072, 5056, 12288, 16384],
          256: [256, 3072, 6400, 9088, 12544], 1024: [1216, 5120, 7232, 13824], 4096: [4096, 12000]}


def _rows(M, K, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    x[:, :: 97] *= 20.0
    x = x.to(dtype)
    if M > 4:
        x[1] = 0
        x[2] = (torch.randn(K, generator=g) * 1e-7).to(dtype)
        x[3, K // 2] = float("inf")
        x[4, 0] = float("nan")
    return x


def _same(a, b):
    """Equal bits, any NaN payload."""
    na, nb = torch.isnan(a), torch.isnan(b)
    assert torch.equal(na, nb)
    assert torch.equal(a.view(torch.int16)[~na], b.view(torch.int16)[~nb])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R", sorted(WIDTHS))
@pytest.mark.parametrize("use_sr,use_perm", [(False, False), (True, False), (False, True), (True, True)])
def test_prepared_rows_equal_the_general_kernel(rt, dev, dtype, R, use_sr, use_perm):
    for K_in in WIDTHS[R]:
        step = max(R, 128)
        K_w = -(-K_in // step) * step if K_in > 64 else K_in
        for M in (1, 7, 700):
            if M == 700 and K_in > 6144:
                continue
            x = _rows(M, K_in, dtype, K_in + M).to(dev)
            g = torch.Generator().manual_seed(K_in)
            sr = rt.prepare_factors(torch.exp(torch.randn(K_in, generator=g) * 0.5).to(dev), dtype) if use_sr else None
            pp = rt.prepare_perm(torch.randperm(K_w, generator=g).to(dev), K_w) if use_perm else None
            kw = dict(rot_size=R, w_in=K_w, smoothrot=sr, perm=pp)
            ref = rt.prepare_activation(x, out=torch.empty(M, K_w + 4, dtype=dtype, device=dev)[:, :K_w], **kw)
            _same(rt.prepare_activation(x, **kw), ref.contiguous())


def test_prepared_rows_strided_and_in_place(rt, dev):
    x = _rows(37, 3072, torch.bfloat16, 5).to(dev)
    ref = rt.prepare_activation(x, rot_size=256)
    wide = torch.zeros(37, 4000, dtype=torch.bfloat16, device=dev)
    wide[:, 8 : 8 + 3072] = x
    out = torch.zeros(37, 3200, dtype=torch.bfloat16, device=dev)
    rt.prepare_activation(wide[:, 8 : 8 + 3072], rot_size=256, out=out[:, :3072])
    _same(out[:, :3072].contiguous(), ref)
    assert not out[:, 3072:].any()
    rt.prepare_activation(x, rot_size=256, out=x)
    _same(x, ref)
