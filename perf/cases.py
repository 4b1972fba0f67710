"""Performance cases: quantized linears of diffusion transformers, from one modulation row to a video block.

A case is one linear layer as the layer code runs it: the activation preparation (SmoothRot divide, block
Hadamard, pad, PermuQuant gather, per-token INT8), or a LayerNorm / RMSNorm fused in front of it, and then the
INT4 or INT8 product with its bias, activation and residual, through the callables of `_hip_runtime`.  Weights are
Gaussian, quantized as the checkpoints hold them; the copies that the drop-in Linear keeps per layer (K-interleaved,
unpacked, staged) are made once in prepare(), by the rules it asks.

kind     "w4a8" (packed INT4 weights, INT8 activations), "w8a8", "w4a16" (INT4 weights, 16-bit activations)
M        tokens;  K_in: input features;  N: output features
rot      Hadamard block, 0 for none;  group: columns per weight scale, 0 for one per output channel
norm     "layer" / "rms" fused in front of the preparation with an adaptive scale and shift, "" for none
factors  SmoothRot factors and a PermuQuant order, as converted checkpoints carry them
act      0 none, 3 GELU (tanh);  residual: an [M, N] tensor added in the epilogue
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys

import torch

_PKG = "comfyui-int-crush_amd"


def _runtime():
    """The package's kernel runtime (the package folder's name has a hyphen)."""
    name = _PKG + "._hip_runtime"
    if name not in sys.modules:
        folder = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), _PKG)
        spec = importlib.util.spec_from_file_location(_PKG, os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[_PKG] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _case(name, kind, M, K_in, N, rot=0, group=128, dtype="bf16", norm="", factors=True, bias=True, act=0,
          residual=False):
    return dict(name=name, kind=kind, M=M, K_in=K_in, N=N, rot=rot, group=group, dtype=dtype, norm=norm,
                factors=factors, bias=bias, act=act, residual=residual)


def listed():
    return [
        # one conditioning vector through a block's modulation layer: weight streaming and launch latency
        _case("w4a8_modulation", "w4a8", 1, 3072, 18432, rot=256),
        # the same layer where the name rule leaves it unrotated, a batch of two
        _case("w4a16_modulation_b2", "w4a16", 2, 3072, 9216, factors=False),
        # a short prompt on an INT8 checkpoint, odd row count, output projection of the text stream
        _case("w8a8_text_77", "w8a8", 77, 4096, 4096, rot=64, group=0, dtype="fp16"),
        # the text stream of a joint block: MLP up behind its adaptive LayerNorm, then MLP down with its residual
        _case("w4a8_text_mlp_up", "w4a8", 512, 3072, 12288, rot=256, norm="layer", act=3),
        _case("w4a8_text_mlp_down", "w4a8", 512, 12288, 3072, rot=256, residual=True),
        # a small image at an odd token count: groups of 64, unpadded head width
        _case("w4a8_ragged_g64", "w4a8", 1357, 2560, 7688, rot=64, group=64, dtype="fp16"),
        # INT8 checkpoint without rotation, attention projection
        _case("w8a8_proj", "w8a8", 4096, 3072, 3072, group=0, dtype="fp16", factors=False, bias=False),
        # image stream: MLP up behind its LayerNorm, MLP down
        _case("w4a8_mlp_up", "w4a8", 4096, 3072, 12288, rot=256, norm="layer", act=3),
        _case("w4a8_mlp_down", "w4a8", 4608, 12288, 3072, rot=256, dtype="fp16", bias=False),
        # the W4A16 mode of a rotated checkpoint (BASELINE config 2's product)
        _case("w4a16_mlp_up", "w4a16", 4608, 3072, 12288, rot=256, dtype="fp16", bias=False),
        # video block at full token count: qkv on an INT8 checkpoint, FFN down on an INT4 one
        _case("w8a8_video_qkv", "w8a8", 32760, 5120, 15360, rot=1024, group=0, dtype="fp16", factors=False),
        _case("w4a8_video_ffn_down", "w4a8", 32760, 13824, 5120, rot=1024, dtype="fp16", factors=False),
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    while True:
        kind = rng.choice(["w4a8", "w4a8", "w8a8", "w4a16"])
        M = _log_int(rng, 1, 32760)
        if M > 16 and rng.random() < 0.5:
            M |= 1
        c = _case("", kind, M, _log_int(rng, 1024, 14336, 64), _log_int(rng, 1024, 18432, 8))
        del c["name"]
        c["rot"] = rng.choice([64, 256, 256, 1024]) if kind == "w4a8" else rng.choice([0, 64, 256, 1024])
        c["group"] = 0 if kind == "w8a8" else rng.choice([128, 128, 128, 64])
        c["dtype"] = rng.choice(["bf16", "fp16"])
        c["norm"] = rng.choice(["", "", "layer", "rms"]) if kind != "w4a16" else ""
        c["factors"] = c["rot"] > 0 and rng.random() < 0.7
        c["bias"] = kind != "w4a16" and rng.random() < 0.7
        c["act"] = 3 if kind != "w4a16" and rng.random() < 0.25 else 0
        c["residual"] = kind != "w4a16" and rng.random() < 0.25
        if M * c["N"] * _width(c) <= 32760 * 5120 * 14336:  # no more than the largest listed
            return c


def _width(c):
    """Columns of the product: the input rounded up to whole Hadamard blocks and to whole 128-column blocks."""
    step = max(128, c["rot"])
    return -(-c["K_in"] // step) * step


def _dtype(c):
    return torch.bfloat16 if c["dtype"] == "bf16" else torch.float16


def _inputs(c, seed):
    """Checkpoint tensors and activations of a case, on the GPU."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    M, K_in, N, K, dt = c["M"], c["K_in"], c["N"], _width(c), _dtype(c)
    t = {}
    x = torch.randn(M, K_in, generator=g, device=dev)
    hot = torch.randperm(K_in, generator=g, device=dev)[: max(1, K_in // 100)]
    x[:, hot] *= 20.0  # outlier channels
    t["x"] = x.to(dt)
    w = torch.randn(N, K, generator=g, device=dev)
    if c["kind"] == "w8a8":
        s = w.abs().amax(1, keepdim=True) / 127.0
        s = (s / math.sqrt(K)).to(torch.float16).float().clamp_min(1e-6)
        t["w"] = (w / (s * math.sqrt(K))).round().clamp(-127, 127).to(torch.int8)
        t["s_w"] = s
    else:
        gs = c["group"] or K
        s = w.reshape(N, K // gs, gs).abs().amax(2) / 7.0
        s = (s / math.sqrt(K)).to(torch.float16).float().clamp_min(1e-6)
        q = (w.reshape(N, K // gs, gs) / (s * math.sqrt(K)).unsqueeze(2)).round().clamp(-8, 7).to(torch.int8)
        q = q.reshape(N, K // 2, 2)
        t["w"] = ((q[:, :, 0] & 15) | ((q[:, :, 1] & 15) << 4)).view(torch.uint8).contiguous()
        t["s_w"] = s.contiguous()
    if c["factors"]:
        t["f"] = torch.exp(torch.randn(K_in, generator=g, device=dev) * 0.5)
        t["perm"] = torch.randperm(K, generator=g, device=dev)
    if c["norm"]:
        t["nw"] = 1.0 + 0.2 * torch.randn(K_in, generator=g, device=dev)
        t["nb"] = 0.2 * torch.randn(K_in, generator=g, device=dev)
    if c["bias"]:
        t["b"] = (0.02 * torch.randn(N, generator=g, device=dev)).to(dt)
    if c["residual"]:
        t["r"] = torch.randn(M, N, generator=g, device=dev).to(dt)
    return t


def prepare(case, seed):
    rt = _runtime()
    t = _inputs(case, seed)
    K, dt = _width(case), _dtype(case)
    M, N, G = case["M"], case["N"], t["s_w"].shape[1]
    st = {"case": case, "x": t["x"], "K": K, "w": t["w"], "s_w": t["s_w"], "b": t.get("b"), "r": t.get("r"),
          "nw": t.get("nw"), "nb": t.get("nb"), "form": "plain",
          "sr": rt.prepare_factors(t.get("f"), dt), "perm": rt.prepare_perm(t.get("perm"), K)}
    # the per-layer weight copies of the drop-in Linear
    if case["kind"] == "w4a8":
        if rt.w4a8_unpacked_pays(M, N, K, G, device=t["x"].device):
            st["w"], st["form"] = rt.unpack_int4_to_int8(t["w"], K), "unpacked"
        else:
            st["w"], st["form"] = rt.int4_interleave_k(t["w"]), "kil"
    elif case["kind"] == "w4a16" and rt.w4a16_staged_pays(M, N, K, G):
        (st["w"], st["s_w"]), st["form"] = rt.w4a16_stage_layout(t["w"], t["s_w"]), "staged"
    return st


def run(state):
    rt, c, st = _runtime(), state["case"], state
    x, dt = st["x"], st["x"].dtype
    if c["kind"] == "w4a16":
        if c["rot"] or c["factors"] or st["K"] != c["K_in"]:
            x = rt.prepare_activation(x, rot_size=c["rot"], w_in=st["K"], smoothrot=st["sr"], perm=st["perm"])
        if st["form"] == "staged":
            return rt.gemm_w4a16_staged(x, st["w"], st["s_w"], bias=st["b"])
        return rt.gemm_w4a16(x, st["w"], st["s_w"], bias=st["b"])
    if c["norm"]:
        q, s_a = rt.norm_rotate_quantize(x, norm=c["norm"], weight=st["nw"], bias=st["nb"], eps=1e-6,
                                         rot_size=c["rot"], w_in=st["K"], smoothrot=st["sr"], perm=st["perm"])
    else:
        q, s_a = rt.rotate_quantize(x, rot_size=c["rot"], w_in=st["K"], smoothrot=st["sr"], perm=st["perm"])
    kw = dict(bias=st["b"], out_dtype=dt, activation=c["act"], residual=st["r"])
    if c["kind"] == "w8a8":
        return rt.fused_int8_gemm_dequant(q, st["w"], st["s_w"], s_a, **kw)
    if st["form"] == "unpacked":
        return rt.gemm_w4a8_unpacked(q, st["w"], st["s_w"], s_a, **kw)
    return rt.gemm_w4a8(q, st["w"], st["s_w"], s_a, kil=True, **kw)


def work(case):
    M, K_in, N, K = case["M"], case["K_in"], case["N"], _width(case)
    weights = N * K if case["kind"] == "w8a8" else N * K // 2
    scales = 4 * N * (K // case["group"] if case["group"] else 1)
    vectors = (8 * K_in + 4 * K if case["factors"] else 0) + (8 * K_in if case["norm"] else 0) + 2 * N * case["bias"]
    rows = 2 * M * K_in + 2 * M * N * (2 if case["residual"] else 1)
    return {"bytes": weights + scales + vectors + rows, "flops": 2.0 * M * N * K}


def tolerance(case):
    # Four times the distance to exact(): the output's rounding (bf16 8 bits, 1.6e-3..1.8e-3 measured; fp16 11 bits,
    # 2.1e-4..3.2e-4, single codes off by one at a rounding boundary among it).  The codes of the same rows are the
    # same whole numbers whatever the order of the sums; behind a norm, statistics summed in another order move a
    # few values across a boundary of the activation type and with them single codes.
    rel = 7e-3 if case["dtype"] == "bf16" else 1.3e-3
    return {"rel": rel * (1.2 if case["norm"] else 1.0), "max": 10 * rel}


def _hadamard(x, R):
    """x [M, K] float64 times the normalized block Hadamard of R = 4^k, base-4 digit by digit."""
    M, K = x.shape
    h = 1
    while h < R:
        v = x.reshape(-1, 4, h)
        x = (0.5 * v.sum(1, keepdim=True) - v.flip(1)).reshape(M, K)
        h *= 4
    return x


def exact(case, seed):
    t = _inputs(case, seed)
    K_in, K, N, dt = case["K_in"], _width(case), case["N"], _dtype(case)
    # weights as the product reads them, K columns in float64
    if case["kind"] == "w8a8":
        w = t["w"].double()
    else:
        b = t["w"].to(torch.int16)
        q = torch.stack((b & 15, b >> 4), 2).reshape(N, K)
        w = torch.where(q > 7, q - 16, q).double().reshape(N, t["s_w"].shape[1], -1)
        s = t["s_w"].unsqueeze(2)
        if case["kind"] == "w4a16":  # the 16-bit weights of that mode
            w = (w * s.to(dt).double()).to(dt).double().reshape(N, K)
        else:
            w = (w * s.double()).reshape(N, K)
    out = torch.empty(case["M"], N, dtype=torch.float64, device=w.device)
    wt = w.t().contiguous()
    del w
    for m0 in range(0, case["M"], 4096):
        x = t["x"][m0 : m0 + 4096].double()
        # each step below rounds to the activation type, as the path defines it
        if case["norm"]:
            if case["norm"] == "layer":
                x = (x - x.mean(1, keepdim=True)) / torch.sqrt(x.var(1, unbiased=False, keepdim=True) + 1e-6)
            else:
                x = x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6)
            x = (x * t["nw"].double() + t["nb"].double()).to(dt).double()
        if case["factors"]:
            x = (x / t["f"].to(dt).double()).to(dt).double()
        x = torch.nn.functional.pad(x, (0, K - K_in))
        if case["rot"]:
            x = _hadamard(x, case["rot"]).to(dt).double()
        if case["factors"]:
            x = x[:, t["perm"]]
        if case["kind"] == "w4a16":
            v = x @ wt
        else:
            s_a = x.abs().amax(1, keepdim=True).clamp_min(1e-8) / 127.0
            v = (x / s_a + 0.5 * torch.sign(x)).trunc() @ wt * s_a
            if case["kind"] == "w8a8":
                v = v * t["s_w"].reshape(1, N).double()
        if case["bias"]:
            v = v + t["b"].double()
        if case["act"] == 3:
            v = 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))
        if case["residual"]:
            v = v + t["r"][m0 : m0 + 4096].double()
        out[m0 : m0 + 4096] = v
    return out
