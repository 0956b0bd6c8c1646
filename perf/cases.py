"""Timed cases of the quantized-linear path: what the blocks of the diffusion models issue through the package's public
entry points (qlinear, weights), from one modulation row to whole images and videos.

A case is a dict of plain values.  `kind` names the call sequence, the other keys its sizes and options.
"""
import importlib
import math

import torch

_pkg = "comfyui-backend-but-rust_amd"
ffi = importlib.import_module(_pkg + ".ffi")
qlinear = importlib.import_module(_pkg + ".qlinear")
weights = importlib.import_module(_pkg + ".weights")

DEV = "cuda:0"
_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_SIZE = {"bf16": 2, "f16": 2, "f32": 4}


def listed():
    return [
        # adaLN modulation of a DiT block: three conditioning rows, one call per block and step
        {"name": "modulation_m3", "kind": "linear", "m": 3, "k": 256, "n": 18432, "rotate": 256, "bias": True, "dtype": "bf16"},
        # a decoder-only text encoder's MLP on a prompt: gate and up as one matrix, weights streamed from HBM
        {"name": "prompt_gate_up_m256", "kind": "linear", "m": 256, "k": 4096, "n": 24576, "rotate": 128, "bias": True, "dtype": "bf16"},
        # the MLP's down projection on a short prompt (77 tokens): few output columns, long K
        {"name": "prompt_down_m77", "kind": "linear", "m": 77, "k": 12288, "n": 4096, "rotate": 128, "bias": False, "dtype": "bf16"},
        # image DiT, 1024x1024 plus 512 text tokens: the MLP's up projection
        {"name": "dit_mlp_up", "kind": "linear", "m": 4608, "k": 3072, "n": 12288, "rotate": 128, "bias": True, "dtype": "bf16"},
        # the same block's way back: SwiGLU inside the quantizer, then the down projection with gate and residual
        {"name": "dit_swiglu_down", "kind": "swiglu_down", "m": 4608, "k": 12288, "n": 3072, "dtype": "bf16"},
        # SDXL transformer level at 1024x1024 with guidance (2 x 4096 rows, 640 wide): LayerNorm, GEGLU up, down + residual
        {"name": "sdxl_feed_forward", "kind": "sd_ff", "m": 8192, "c": 640, "dtype": "f16"},
        # joint attention of the image DiT: per-head RMSNorm and rotary embedding fused into the quantizers
        {"name": "dit_joint_attention", "kind": "attn", "form": "norm_rope", "b": 1, "lq": 4608, "lk": 4608, "h": 24, "d": 128, "dtype": "bf16"},
        # SDXL self-attention at the 64x64 latent level, head dim 64, half precision
        {"name": "sdxl_self_attention", "kind": "attn", "form": "plain", "b": 2, "lq": 4096, "lk": 4096, "h": 10, "d": 64, "dtype": "f16"},
        # video DiT FFN up with packed 6-bit weights and fp32 scales per 128 along K (rows already quantized: the
        # quantizer's output feeds several linears)
        {"name": "video_w6_group_up", "kind": "w6_group", "m": 8192, "k": 5120, "n": 13824, "dtype": "bf16"},
        # a linear stored in the two-plane W6 checkpoint form, run the way weights.py runs it
        {"name": "w6_checkpoint_down", "kind": "w6_linear", "m": 2048, "k": 14336, "n": 5376, "dtype": "bf16"},
        # baking an adapter into int8 weights: back to the original basis, and the patched weight to codes again
        {"name": "bake_int8", "kind": "bake_int8", "n": 12288, "k": 3072, "seed": 12345, "dtype": "bf16"},
        # baking an adapter into W6 weights: least-squares steps, stochastic rounding, packing; and the decode of the result
        {"name": "bake_w6", "kind": "bake_w6", "n": 5376, "k": 5376, "seed": 777, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    return max(lo, _log(rng, lo, hi) // step * step)


def draw(rng):
    """One more case of the ranges above: any row count, widths in the steps that the formats allow."""
    kind = rng.choice(("linear", "linear", "linear", "swiglu_down", "sd_ff", "attn", "attn", "w6_group", "w6_linear", "bake_int8", "bake_w6"))
    if kind == "linear":
        while True:
            m, k, n = _log(rng, 1, 8192), _mult(rng, 256, 14336, 256), _mult(rng, 96, 24576, 8)
            if m * k * n <= 3e11 and k * n >= 2 ** 18:
                break
        dt = rng.choice(("bf16", "bf16", "bf16", "f32"))
        return {"kind": kind, "m": m, "k": k, "n": n, "rotate": rng.choice((0, 128, 256, 256)), "bias": rng.random() < 0.5, "dtype": dt}
    if kind == "swiglu_down":
        while True:
            m, k, n = _log(rng, 128, 8192), _mult(rng, 2048, 16384, 256), _mult(rng, 1024, 6144, 32)
            if m * k * n <= 3e11:
                break
        return {"kind": kind, "m": m, "k": k, "n": n, "dtype": "bf16"}
    if kind == "sd_ff":
        return {"kind": kind, "m": _log(rng, 256, 16384), "c": 64 * rng.randint(5, 20), "dtype": "f16"}
    if kind == "attn":
        while True:
            b, d = rng.choice((1, 1, 2)), rng.choice((64, 128, 128))
            lq, h = _log(rng, 256, 8192), rng.randint(5, 32)
            form = "plain" if d == 64 else rng.choice(("plain", "norm_rope", "key_bias"))
            lk = lq if form == "norm_rope" else rng.choice((lq, lq, rng.randint(77, 512)))
            if b * h * lq * lk * d <= 1.2e11:
                break
        dt = rng.choice(("bf16", "f16")) if form == "plain" else "bf16"
        return {"kind": kind, "form": form, "b": b, "lq": lq, "lk": lk, "h": h, "d": d, "dtype": dt}
    if kind == "w6_group":
        while True:
            m, k, n = _log(rng, 64, 8192), _mult(rng, 1024, 13824, 128), _mult(rng, 1024, 13824, 32)
            if m * k * n <= 5e11:
                break
        return {"kind": kind, "m": m, "k": k, "n": n, "dtype": "bf16"}
    if kind == "w6_linear":
        while True:
            m, k, n = _log(rng, 64, 8192), _mult(rng, 1024, 14336, 256), _mult(rng, 1024, 28672, 32)
            if m * k * n <= 4e11:
                break
        return {"kind": kind, "m": m, "k": k, "n": n, "dtype": "bf16"}
    while True:
        n, k = _log(rng, 512, 24576), _mult(rng, 512, 16384, 256)
        if n * k <= (6e7 if kind == "bake_int8" else 3e7):
            break
    return {"kind": kind, "n": n, "k": k, "seed": rng.choice((0, rng.randint(1, 1 << 30))), "dtype": rng.choice(("bf16", "f32")) if kind == "bake_int8" else "bf16"}


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _acts(g, m, k, dtype):
    """Activations with heavy-tailed channels: normal rows times a per-channel Student-t(3) scale."""
    c = torch.randn(k, device=DEV, generator=g) / torch.sqrt(sum(torch.randn(k, device=DEV, generator=g) ** 2 for _ in range(3)) / 3.0)
    x = torch.randn(m, k, device=DEV, generator=g)
    return x.mul_(c.clamp_(-30, 30)).to(dtype)


def _codes(g, m, k):
    return torch.randint(-127, 128, (m, k), dtype=torch.int8, device=DEV, generator=g)


def _scales(g, n, lo=1e-3, hi=1e-2):
    return lo + (hi - lo) * torch.rand(n, device=DEV, generator=g)


def _vec(g, n, dtype, gain=0.02, at=0.0):
    return (at + gain * torch.randn(n, device=DEV, generator=g)).to(dtype)


def prepare(case, seed):
    g, kind, dt = _gen(seed), case["kind"], _DT[case["dtype"]]
    s = {"kind": kind, "dt": dt}
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        s.update(x=_acts(g, m, k, dt), W=_codes(g, n, k), ws=_scales(g, n), bias=_vec(g, n, dt) if case["bias"] else None, rotate=case["rotate"])
    elif kind == "swiglu_down":
        m, k, n = case["m"], case["k"], case["n"]
        s.update(gu=_acts(g, m, 2 * k, dt), k=k, W=_codes(g, n, k), ws=_scales(g, n), rscale=_vec(g, n, dt, 0.3), resid=torch.randn(m, n, device=DEV, generator=g).to(dt))
    elif kind == "sd_ff":
        m, c = case["m"], case["c"]
        i = 4 * c
        s.update(x=torch.randn(m, c, device=DEV, generator=g).to(dt), ln_w=_vec(g, c, torch.float32, 0.1, 1.0), ln_b=_vec(g, c, torch.float32),
                 W1=_codes(g, 2 * i, c), ws1=_scales(g, 2 * i, 1e-4, 1e-3), b1=_vec(g, 2 * i, dt),
                 W2=_codes(g, c, i), ws2=_scales(g, c, 1e-4, 1e-3), b2=_vec(g, c, dt), ones=torch.ones(c, device=DEV, dtype=dt),
                 rot1=256 if c % 256 == 0 else 64, rot2=256 if i % 256 == 0 else 64)
    elif kind == "attn":
        b, lq, lk, h, d = (case[v] for v in ("b", "lq", "lk", "h", "d"))
        if lq == lk:   # heads of one packed projection, as the block's QKV linear leaves them
            qkv = torch.randn(b, lq, 3, h, d, device=DEV, generator=g).to(dt)
            q, k, v = qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
        else:          # cross-attention: q from the image, k and v from the text
            q = torch.randn(b, lq, h, d, device=DEV, generator=g).to(dt)
            kv = torch.randn(b, lk, 2, h, d, device=DEV, generator=g).to(dt)
            k, v = kv[:, :, 0], kv[:, :, 1]
        s.update(form=case["form"], q=q, k=k, v=v, scale=d ** -0.5)
        if case["form"] == "norm_rope":
            pos = torch.arange(max(lq, lk), device=DEV, dtype=torch.float32)[:, None]
            ang = pos * torch.exp(-9.2 * torch.arange(d // 2, device=DEV, dtype=torch.float32) / (d // 2))[None, :]
            s.update(qw=_vec(g, d, torch.float32, 0.1, 1.0), kw=_vec(g, d, torch.float32, 0.1, 1.0), rope=torch.stack((torch.cos(ang), torch.sin(ang)), -1).contiguous())
        if case["form"] == "key_bias":
            bias = torch.zeros(lk, device=DEV)
            bias[torch.randint(0, lk, (max(1, lk // 16),), device=DEV, generator=g)] = 0.6
            s.update(key_bias=bias)
            nws = ffi.lib.gpu_int8_attn_key_bias_workspace(b, h, h, lq, lk)
        else:
            nws = ffi.lib.gpu_int8_attn_workspace_d(b, h, h, lq, lk, d)
        s.update(ws=torch.empty(nws, dtype=torch.uint8, device=DEV))
    elif kind == "w6_group":
        m, k, n = case["m"], case["k"], case["n"]
        u = torch.randint(1, 64, (n, k // 4, 4), dtype=torch.int32, device=DEV, generator=g)   # code + 32
        w = u[..., 0] | (u[..., 1] << 6) | (u[..., 2] << 12) | (u[..., 3] << 18)
        s.update(packed=torch.stack((w & 255, (w >> 8) & 255, w >> 16), dim=-1).to(torch.uint8).reshape(n, k // 4 * 3).contiguous(), A=_codes(g, m, k),
                 xs=_scales(g, m, 0.01, 0.11), sw=_scales(g, n * (k // 128)).view(n, k // 128), bias=_vec(g, n, dt))
    elif kind == "w6_linear":
        m, k, n = case["m"], case["k"], case["n"]
        packed = torch.randint(0, 256, (n, k // 4 * 3), dtype=torch.uint8, device=DEV, generator=g)
        e = torch.randint(6, 9, (n, k // 32), device=DEV, generator=g) * 8 + torch.randint(0, 8, (n, k // 32), device=DEV, generator=g)   # e4m3 in [0.5, 3.75]
        s.update(x=_acts(g, m, k, dt), lin=weights.Linear("w6", n, k, packed, _scales(g, n), e.to(torch.uint8), None))
    elif kind == "bake_int8":
        n, k = case["n"], case["k"]
        s.update(q=_codes(g, n, k), ws=_scales(g, n), patched=(0.02 * torch.randn(n, k, device=DEV, generator=g)).to(dt), seed=case["seed"])
    elif kind == "bake_w6":
        n, k = case["n"], case["k"]
        s.update(patched=(0.02 * torch.randn(n, k, device=DEV, generator=g)).to(dt), seed=case["seed"], n=n, k=k)
    else:
        raise ValueError(kind)
    return s


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return qlinear.linear_w8a8(s["x"], s["W"], s["ws"], s["bias"], s["rotate"])
    if kind == "swiglu_down":
        q, xs = qlinear.quant_rows_pro(s["gu"], ffi.PRO_SWIGLU, s["k"], 1, up_offset=s["k"])
        return qlinear.int8_gemm_residual(q, s["W"], xs, s["ws"], None, s["rscale"], s["resid"])
    if kind == "sd_ff":
        q, xs = qlinear.sd_ln_quant_rows(s["x"], s["ln_w"], s["ln_b"], 1e-5, s["rot1"])
        up = qlinear.int8_gemm(q, s["W1"], xs, s["ws1"], s["b1"], s["dt"])
        q, xs = qlinear.sd_geglu_quant_rows(up, s["rot2"])
        return qlinear.int8_gemm_residual(q, s["W2"], xs, s["ws2"], s["b2"], s["ones"], s["x"])
    if kind == "attn":
        if s["form"] == "norm_rope":
            return qlinear.int8_attn_norm_rope(s["q"], s["k"], s["v"], s["scale"], s["qw"], s["kw"], 1e-6, s["rope"], 1, s["ws"])
        if s["form"] == "key_bias":
            return qlinear.int8_attn_key_bias(s["q"], s["k"], s["v"], s["scale"], s["key_bias"], s["ws"])
        return qlinear.int8_attn(s["q"], s["k"], s["v"], s["scale"], s["ws"])
    if kind == "w6_group":
        return qlinear.w6a8_group_gemm(s["A"], s["packed"], s["xs"], s["sw"], s["bias"])
    if kind == "w6_linear":
        return weights.forward(s["lin"], s["x"])
    if kind == "bake_int8":
        return qlinear.convrot_dequant(s["q"], s["ws"], s["dt"]), qlinear.convrot_requant(s["patched"], s["seed"])
    packed, s_rel, s_ch = qlinear.w6_requant(s["patched"], s["seed"])
    return packed, s_rel, s_ch, qlinear.w6_decode(packed, s_rel, s["n"], s["k"], 32)


def work(case):
    """Bytes each input and output needs once (intermediates that stay between two calls of one pass are not counted)
    and operations of the matrix products."""
    kind, e = case["kind"], _SIZE[case["dtype"]]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": m * k * e + n * k + n * 4 + (n * e if case["bias"] else 0) + m * n * e, "flops": 2.0 * m * n * k}
    if kind == "swiglu_down":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": m * 2 * k * e + n * k + n * (4 + e) + 2 * m * n * e, "flops": 2.0 * m * n * k}
    if kind == "sd_ff":
        m, c = case["m"], case["c"]
        return {"bytes": 2 * m * c * e + 12 * c * c + 8 * c * (4 + e) + c * (12 + 2 * e), "flops": 24.0 * m * c * c}
    if kind == "attn":
        b, lq, lk, h, d = (case[v] for v in ("b", "lq", "lk", "h", "d"))
        return {"bytes": 2 * b * h * d * e * (lq + lk), "flops": 4.0 * b * h * lq * lk * d}
    if kind == "w6_group":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": m * k + m * 4 + n * k * 3 // 4 + n * (k // 128) * 4 + n * e + m * n * e, "flops": 2.0 * m * n * k}
    if kind == "w6_linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": m * k * e + n * k * 3 // 4 + n * (k // 32) + n * 4 + m * n * 2, "flops": 2.0 * m * n * k}
    n, k = case["n"], case["k"]
    if kind == "bake_int8":
        return {"bytes": n * k * (2 + 2 * e) + 8 * n, "flops": 0.0}
    return {"bytes": n * k * e + n * k * 3 // 4 + n * (k // 32) + 4 * n + n * k, "flops": 0.0}


def tolerance(case):
    """About four times what is seen against the same path in 64 bits (bf16 outputs 1.7e-3, f32 outputs 4.6e-5: the last
    rounding, and codes on the other side of a tie); half-precision outputs four times the rounding to half.  Attention
    differs from an implementation with a correctly rounded exp2 by 2e-5 before that rounding.  Codes, packed bytes and
    scales of the weight formats are exact."""
    if case["kind"] in ("bake_int8", "bake_w6"):
        return "exact"
    return {"rel": {"bf16": 7e-3, "f16": 1e-3, "f32": 2e-4}[case["dtype"]]}
