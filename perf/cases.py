"""The workloads this library is timed and checked on, each through its public entry points.

A case is a dict of plain values. Its "op" says which call of a DiT block or of the text
and vision encoders in front of it the case stands for:

  attn       flash_attn: BF16 attention (causal prefill, vision encoder, image tokens)
  sage       flash_attn_fp8: INT8/FP8 attention on normalised Q and K, prologue included
  sage_rope  flash_attn_fp8_norm_rope: the same from the raw fused QKV projection
  linear     quantize_blockscaled of the activations, then gemm_blockscaled
  norm_rope  head_norm_rope of Q and of K out of the fused QKV projection

Sizes are those of the benchmark configurations and of the tests (24 heads of 128 with 4352
or 12544 tokens, 40 heads with 32760, 32 query heads on 8 key heads, 16 heads of 72, linears
of 3072, 4096 and 12288 features), and draw() spreads over the ranges around them.
"""
from __future__ import annotations

import math

import torch

from miroxen_amd.attention import (ROPE_HALF, ROPE_INTERLEAVED, AttnParams, flash_attn, flash_attn_fp8,
                                   flash_attn_fp8_norm_rope, flash_attn_fp8_workspace, head_norm_rope)
from miroxen_amd.blockscale import QMat, QMode, gemm_blockscaled, qdata_bytes, qscale_bytes, quantize_blockscaled

EPS = 1e-6
DEV = "cuda:0"


def _attn(name, Sq, Skv, Hq, Hkv, D, causal=0, q_offset=0, text=0, text_valid=0, pad=0):
    """pad: elements after the heads of a token in Q, K and V (a padded row stride)."""
    return {"name": name, "op": "attn", "Sq": Sq, "Skv": Skv, "Hq": Hq, "Hkv": Hkv, "D": D, "causal": causal,
            "q_offset": q_offset, "text": text, "text_valid": text_valid, "pad": pad}


def _sage(name, S, H, D=128, text=0, text_valid=0, outliers=8):
    return {"name": name, "op": "sage", "S": S, "H": H, "D": D, "text": text, "text_valid": text_valid,
            "outliers": outliers}


def _sage_rope(name, S, H, rot, mode, text=0, text_valid=0):
    return {"name": name, "op": "sage_rope", "S": S, "H": H, "D": 128, "rot": rot, "mode": mode, "text": text,
            "text_valid": text_valid}


def _linear(name, mode, M, N, K):
    return {"name": name, "op": "linear", "mode": mode, "M": M, "N": N, "K": K}


def _norm_rope(name, S, H, D, rot, mode):
    return {"name": name, "op": "norm_rope", "S": S, "H": H, "D": D, "rot": rot, "mode": mode}


def listed():
    return [
        # the prompt of one image through the text encoder: the smallest attention calls
        _attn("prompt_causal", 333, 333, 32, 8, 128, causal=1),
        # a long prompt prefilled behind 117 cached tokens
        _attn("prefill_causal_offset", 2048, 2165, 32, 8, 128, causal=1, q_offset=117),
        # one reference image through the vision encoder: heads of 72 channels, token rows
        # padded to whole 64-byte lines
        _attn("vision_d72", 4096, 4096, 16, 16, 72, pad=32),
        # joint attention of a 1024 x 1024 image in BF16, 200 of 256 text slots in use
        _attn("image_bf16", 4352, 4352, 24, 24, 128, text=256, text_valid=200),
        # a 512 x 512 image's joint attention, quantized
        _sage("small_image_fp8", 1088, 24),
        # the 1024 x 1024 image's joint attention, quantized
        _sage("image_fp8", 4352, 24, text=256, text_valid=200),
        # image editing with two reference images in the sequence
        _sage("edit_fp8", 12544, 24, text=256, text_valid=180, outliers=0),
        # a video's packed sequence, from the QKV projection, rotary half of the channels
        _sage_rope("video_rope_fp8", 32760, 40, 64, "half"),
        # the text stream's projections: few rows, all of the weights
        _linear("text_linear_mxfp8", "mxfp8", 256, 3072, 3072),
        # the widest linear at the image stream's largest batch of rows
        _linear("image_linear_mxfp8", "mxfp8", 8192, 12288, 4096),
        # the MLP's second linear of the image stream in 4 bits
        _linear("image_linear_nvfp4", "nvfp4", 4096, 3072, 12288),
        # Q and K of the image stream before BF16 attention
        _norm_rope("image_norm_rope", 4352, 24, 128, 128, "interleaved"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _text(rng, S):
    """Text slots at the front of an image's sequence and how many of them are in use."""
    if S < 512 or rng.random() < 0.4:
        return 0, 0
    return 256, rng.randint(1, 256)


def draw(rng):
    op = rng.choice(("causal", "vision", "image", "sage", "sage", "sage_rope", "linear", "linear", "linear", "norm_rope"))
    if op == "causal":
        S, off = _log(rng, 17, 4096), rng.choice((0, 0, rng.randint(1, 1024)))
        hq, hkv = rng.choice(((32, 8), (16, 8), (64, 8), (32, 32)))
        c = _attn("", S, S + off, hq, hkv, 128, causal=1, q_offset=off)
    elif op == "vision":
        S = _log(rng, 200, 12000)
        H = rng.choice((8, 16))
        c = _attn("", S, S, H, H, rng.choice((64, 72, 72)), pad=32)
    elif op == "image":
        S, H = _log(rng, 300, 12544), rng.choice((24, 40))
        text, valid = _text(rng, S)
        c = _attn("", S, S, H, H, 128, text=text, text_valid=valid)
    elif op == "sage":
        S = _log(rng, 300, 16384)
        text, valid = _text(rng, S)
        c = _sage("", S, rng.choice((24, 40)), rng.choice((128, 128, 128, 64)), text, valid, rng.choice((0, 8)))
    elif op == "sage_rope":
        S = _log(rng, 500, 20000)
        text, valid = _text(rng, S)
        rot, mode = rng.choice(((64, "half"), (128, "interleaved"), (128, "half")))
        c = _sage_rope("", S, rng.choice((24, 40)), rot, mode, text, valid)
    elif op == "linear":
        feats = (1024, 3072, 4096, 5120, 12288)
        N = rng.choice(feats) if rng.random() < 0.7 else _log(rng, 64, 12288)
        K = rng.choice(feats) if rng.random() < 0.7 else 32 * _log(rng, 8, 384)
        c = _linear("", rng.choice(("mxfp8", "mxfp8", "nvfp4")), _log(rng, 1, 8192), N, K)
    else:
        H, D, rot, mode = rng.choice(((24, 128, 128, "interleaved"), (40, 128, 64, "half"), (32, 128, 128, "half"),
                                      (16, 72, 72, "half")))
        c = _norm_rope("", _log(rng, 64, 32760), H, D, rot, mode)
    del c["name"]
    return c


# ---------------- inputs ----------------

def _randn(shape, seed, scale=1.0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * scale


def _rand(shape, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float32)


def _head_rows(S, H, D, seed):
    """Q or K as head_norm_rope leaves them: rows of unit RMS times a gain per channel."""
    x = _randn((S, H, D), seed)
    x *= torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return x * (_rand((D,), seed + 1) + 0.5)


def _padded(x, pad):
    """x [S, H, D] as the first H * D elements of rows with `pad` more behind them."""
    S, H, D = x.shape
    rows = torch.zeros(S, H * D + pad, dtype=x.dtype, device=DEV)
    rows[:, : H * D] = x.view(S, H * D)
    return rows[:, : H * D].view(S, H, D) if pad else x


def _outliers(k, n, seed):
    """A constant offset in n channels of each head, as K shows it in diffusion transformers."""
    S, H, D = k.shape
    if not n:
        return k
    off = torch.zeros(H, D, device=DEV)
    at = _rand((H, D), seed).argsort(-1)[:, :n]
    off.scatter_(1, at, _randn((H, n), seed + 1, 2.0))
    return k + off


def _mask(S, text, valid, seed):
    if not text:
        return None
    m = torch.ones(S, dtype=torch.uint8, device=DEV)
    m[:text] = 0
    m[_rand((text,), seed).argsort()[:valid]] = 1
    return m


def _qkv(case, seed):
    b = seed * 100
    if case["op"] == "attn":
        Sq, Skv, Hq, Hkv, n = case["Sq"], case["Skv"], case["Hq"], case["Hkv"], 0
    else:
        Sq = Skv = case["S"]
        Hq = Hkv = case["H"]
        n = case["outliers"]
    D = case["D"]
    q = _head_rows(Sq, Hq, D, b + 1).to(torch.bfloat16)
    k = _outliers(_head_rows(Skv, Hkv, D, b + 3), n, b + 5).to(torch.bfloat16)
    v = _randn((Skv, Hkv, D), b + 7).to(torch.bfloat16)
    q, k, v = (_padded(x, case.get("pad", 0)) for x in (q, k, v))
    return q, k, v, _mask(Skv, case["text"], case["text_valid"], b + 8)


def _rope_tables(S, rot):
    freq = 10000.0 ** (-torch.arange(rot // 2, device=DEV, dtype=torch.float64) * 2 / rot)
    ang = torch.arange(S, device=DEV, dtype=torch.float64)[:, None] * freq
    return ang.cos().float().contiguous(), ang.sin().float().contiguous()


def _projection(case, seed):
    """The fused QKV projection [S, 3, H, D], the norms' weights and the rotary tables."""
    S, H, D, b = case["S"], case["H"], case["D"], seed * 100
    t = _randn((S, 3, H, D), b + 1, 1.5).to(torch.bfloat16)
    return t, _rand((D,), b + 2) + 0.5, _rand((D,), b + 3) + 0.5, *_rope_tables(S, case["rot"])


def _operands(case, seed):
    """Activations with a few large values among them, and the weights of a linear."""
    M, N, K, b = case["M"], case["N"], case["K"], seed * 100
    x = _randn((M, K), b + 1)
    x = torch.where(_rand((M, K), b + 2) < 0.02, x * 20, x).to(torch.bfloat16)
    return x, _randn((N, K), b + 3, 0.02).to(torch.bfloat16)


MODES = {"half": ROPE_HALF, "interleaved": ROPE_INTERLEAVED}
QMODES = {"mxfp8": QMode.MXFP8, "nvfp4": QMode.NVFP4}


def _qmat(mode, rows, K):
    return QMat(torch.empty(qdata_bytes(mode, rows, K), dtype=torch.uint8, device=DEV),
                torch.empty(qscale_bytes(mode, rows, K), dtype=torch.uint8, device=DEV),
                torch.zeros(1, dtype=torch.float32, device=DEV) if mode == QMode.NVFP4 else None)


def prepare(case, seed):
    op = case["op"]
    if op == "attn":
        q, k, v, m = _qkv(case, seed)
        p = AttnParams(Sq=case["Sq"], Skv=case["Skv"], Hq=case["Hq"], Hkv=case["Hkv"], D=case["D"],
                       causal=case["causal"], q_offset=case["q_offset"], q_stride=q.stride(0),
                       kv_stride=k.stride(0), kv_valid=m)
        o = torch.empty(q.shape, dtype=torch.bfloat16, device=DEV)
        return {"op": op, "q": q, "k": k, "v": v, "o": o, "p": p}
    if op == "sage":
        q, k, v, m = _qkv(case, seed)
        p = AttnParams(Sq=case["S"], Skv=case["S"], Hq=case["H"], Hkv=case["H"], D=case["D"], kv_valid=m)
        ws = torch.empty(flash_attn_fp8_workspace(p), dtype=torch.uint8, device=DEV)
        return {"op": op, "q": q, "k": k, "v": v, "o": torch.empty_like(q), "p": p, "ws": ws}
    if op == "sage_rope":
        S, H, D = case["S"], case["H"], case["D"]
        t, qw, kw, cos, sin = _projection(case, seed)
        m = _mask(S, case["text"], case["text_valid"], seed * 100 + 8)
        p = AttnParams(Sq=S, Skv=S, Hq=H, Hkv=H, D=D, q_stride=3 * H * D, kv_stride=3 * H * D, o_stride=H * D,
                       kv_valid=m)
        ws = torch.empty(flash_attn_fp8_workspace(p), dtype=torch.uint8, device=DEV)
        o = torch.empty(S, H, D, dtype=torch.bfloat16, device=DEV)
        return {"op": op, "t": t, "qw": qw, "kw": kw, "cos": cos, "sin": sin, "rot": case["rot"],
                "mode": MODES[case["mode"]], "o": o, "p": p, "ws": ws}
    if op == "linear":
        M, N, K, mode = case["M"], case["N"], case["K"], QMODES[case["mode"]]
        x, w = _operands(case, seed)
        W, X = _qmat(mode, N, K), _qmat(mode, M, K)
        quantize_blockscaled(mode, w, K, N, K, W)
        return {"op": op, "mode": mode, "x": x, "W": W, "X": X, "M": M, "N": N, "K": K,
                "y": torch.empty(M, N, dtype=torch.bfloat16, device=DEV)}
    t, qw, kw, cos, sin = _projection(case, seed)
    S, H, D = case["S"], case["H"], case["D"]
    q, k = (torch.empty(S, H, D, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    return {"op": op, "t": t, "qw": qw, "kw": kw, "cos": cos, "sin": sin, "rot": case["rot"],
            "mode": MODES[case["mode"]], "S": S, "H": H, "D": D, "q": q, "k": k}


def run(s):
    op = s["op"]
    if op == "attn":
        flash_attn(s["q"], s["k"], s["v"], s["o"], s["p"])
        return s["o"]
    if op == "sage":
        flash_attn_fp8(s["q"], s["k"], s["v"], s["o"], s["p"], s["ws"])
        return s["o"]
    if op == "sage_rope":
        t = s["t"]
        flash_attn_fp8_norm_rope(t[:, 0], t[:, 1], t[:, 2], s["o"], s["p"], s["qw"], s["kw"], EPS, s["cos"], s["sin"],
                                 s["rot"], s["mode"], s["ws"])
        return s["o"]
    if op == "linear":
        mode, M, N, K, X = s["mode"], s["M"], s["N"], s["K"], s["X"]
        quantize_blockscaled(mode, s["x"], K, M, K, X)
        gemm_blockscaled(mode, s["W"], X, s["y"], N, M, N, K)
        return {"y": s["y"], "xq": X.q, "xsf": X.sf}
    S, H, D = s["S"], s["H"], s["D"]
    for i, (w, out) in enumerate(((s["qw"], s["q"]), (s["kw"], s["k"]))):
        head_norm_rope(s["t"], S, 3 * H * D, i * H * D, H, D, w, EPS, s["cos"], s["sin"], s["rot"], s["mode"], out)
    return {"q": s["q"], "k": s["k"]}


def _pairs(case):
    """(query, key) pairs of one head that the softmax takes in."""
    if case["op"] != "attn":
        return case["S"] * (case["S"] - case["text"] + case["text_valid"])
    Sq, Skv = case["Sq"], case["Skv"]
    if case["causal"]:
        return sum(min(Skv, case["q_offset"] + i + 1) for i in range(Sq))
    return Sq * (Skv - case["text"] + case["text_valid"])


def work(case):
    op = case["op"]
    if op == "attn":
        D = case["D"]
        return {"bytes": 2 * D * 2 * (case["Sq"] * case["Hq"] + case["Skv"] * case["Hkv"]),
                "flops": 4 * case["Hq"] * D * _pairs(case)}
    if op in ("sage", "sage_rope"):
        n = case["S"] * case["H"] * case["D"]
        tables = 4 * case["S"] * case["rot"] if op == "sage_rope" else 0
        return {"bytes": 8 * n + tables, "flops": 4 * case["H"] * case["D"] * _pairs(case)}
    if op == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        per = 1 + 1 / 32 if case["mode"] == "mxfp8" else 0.5 + 1 / 16
        return {"bytes": 2 * M * K + per * (M * K + N * K) + 2 * M * N, "flops": 2 * M * N * K}
    n = case["S"] * case["H"] * case["D"]
    return {"bytes": 8 * n + 4 * case["S"] * case["rot"], "flops": 2 * 10 * n}


def tolerance(case):
    # BF16 outputs are off the exact values by their own rounding and by that of the
    # probabilities (measured 1.7e-3 for the linears and the norm, 2.0e-3 to 2.3e-3 for
    # attention): about four times that. The quantized bytes of a linear are exact.
    if case["op"] in ("attn", "linear", "norm_rope"):
        return {"rel": 8e-3}
    # Probabilities in e4m3 have three bits of mantissa and put the result 4.0 % off exact
    # attention. With the key tiles taken in another order every one of them rounds anew
    # (the running maximum moves): 3.7 % apart. The bound lies below that, so an
    # implementation keeps the order of the tiles and the rule of the maximum.
    return {"rel": 3e-2}


# ---------------- the same in 64 bits ----------------

def _attention64(q, k, v, causal=False, off=0, mask=None):
    Sq, Hq, D = q.shape
    Skv, Hkv = k.shape[:2]
    out = torch.empty(Sq, Hq, D, dtype=torch.float64, device=DEV)
    step = max(1, (1 << 27) // Skv)
    j = torch.arange(Skv, device=DEV)
    for h in range(Hq):
        g = h // (Hq // Hkv)
        kh, vh = k[:, g].double().t().contiguous(), v[:, g].double().contiguous()
        for a in range(0, Sq, step):
            s = q[a:a + step, h].double() @ kh
            s *= 1 / math.sqrt(D)
            if mask is not None:
                s.masked_fill_(mask == 0, -math.inf)
            if causal:
                i = torch.arange(a, a + s.shape[0], device=DEV)[:, None]
                s.masked_fill_(j > off + i, -math.inf)
            s -= s.amax(-1, keepdim=True)
            s.exp_()
            out[a:a + step, h] = (s @ vh) / s.sum(-1, keepdim=True)
    return out


def _norm_rope64(x, w, cos, sin, rot, mode):
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    c, s = cos.double()[:, None], sin.double()[:, None]
    r = x[..., :rot]
    if mode == "interleaved":
        a, b = r[..., 0::2], r[..., 1::2]
        r = torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)
    else:
        a, b = r[..., : rot // 2], r[..., rot // 2:]
        r = torch.cat((a * c - b * s, b * c + a * s), -1)
    return torch.cat((r, x[..., rot:]), -1)


def _mxfp8_64(x):
    """The values that MXFP8 holds for x: e4m3 times the smallest power of two that takes a
    block of 32 to at most 448."""
    b = x.float().reshape(-1, 32)
    mant, ex = torch.frexp(b.abs().amax(-1, keepdim=True) / 448.0)
    e = torch.where(mant == 0.5, ex - 1, ex).clamp(-127, 127)
    e = torch.where(mant == 0, torch.full_like(e, -127), e).double()
    q = (b.double() * torch.exp2(-e)).clamp(-448, 448).float().to(torch.float8_e4m3fn)
    return (q.double() * torch.exp2(e)).reshape(x.shape)


def _nvfp4_64(x):
    """The values that NVFP4 holds for x: e2m1 times an e4m3 scale per 16 times amax / 2688."""
    b = x.float().reshape(-1, 16)
    amax = b.abs().amax()
    g = amax / 2688.0 if float(amax) > 0 else torch.ones_like(amax)
    se = (b.abs().amax(-1, keepdim=True) * (1.0 / (6.0 * g))).clamp(max=448).to(torch.float8_e4m3fn).float()
    sd = se * g
    t = b * torch.where(sd > 0, 1.0 / sd, torch.zeros_like(sd))
    a = t.abs().clamp(max=6)
    step = torch.where(a < 2, 0.5, torch.where(a < 4, 1.0, 2.0))
    code = torch.round(a / step) * step * torch.sign(t)
    return (code.double() * se.double() * g.double()).reshape(x.shape)


def exact(case, seed):
    op = case["op"]
    if op == "attn":
        q, k, v, m = _qkv(case, seed)
        return _attention64(q, k, v, bool(case["causal"]), case["q_offset"], m)
    if op == "sage":
        q, k, v, m = _qkv(case, seed)
        return _attention64(q, k, v, mask=m)
    if op == "sage_rope":
        t, qw, kw, cos, sin = _projection(case, seed)
        m = _mask(case["S"], case["text"], case["text_valid"], seed * 100 + 8)
        q, k = (_norm_rope64(t[:, i], w, cos, sin, case["rot"], case["mode"]).to(torch.bfloat16)
                for i, w in ((0, qw), (1, kw)))
        return _attention64(q, k, t[:, 2], mask=m)
    if op == "linear":
        x, w = _operands(case, seed)
        held = _mxfp8_64 if case["mode"] == "mxfp8" else _nvfp4_64
        return {"y": held(x) @ held(w).t().contiguous(), "xq": None, "xsf": None}
    t, qw, kw, cos, sin = _projection(case, seed)
    return {"q": _norm_rope64(t[:, 0], qw, cos, sin, case["rot"], case["mode"]),
            "k": _norm_rope64(t[:, 1], kw, cos, sin, case["rot"], case["mode"])}
