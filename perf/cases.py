"""The performance cases of the denoising / autoregressive path.

Each case is one piece of the work that a program has the library do, called as a program calls
it: through the C ABI's entry points (diffuse-cpp_amd/dfx.py) on device buffers, or, for whole
passes, through a model and its context.  The kinds:

  mlp      the FFN block of one layer: RMSNorm + conversion, gate|up GEMM with SwiGLU, conversion,
           down GEMM + residual
  attn     the attention block of one layer: RMSNorm + conversion, Q|K|V GEMM with RoPE and the
           cache store, attention over the cache, conversion, O GEMM + residual
  head     the end of a denoising step: final RMSNorm, vocab GEMM, row statistics, selection
  sampler  row statistics and selection over logits that are there already
  model    whole passes of a small model with host tokens in and host logits out

Shapes are the benchmark's architectures (dfx.LLADA_8B, dfx.DREAM_7B) and the tests' small one.
Weights are random N(0, 0.02), encoded on the GPU into the library's device layout
(include/dfx.h); activations have a per-channel spread, as residual streams have.
"""
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "diffuse-cpp_amd"))
import dfx  # noqa: E402

ARCH = {"llada-8b": dfx.LLADA_8B, "dream-7b": dfx.DREAM_7B}
TYPE = {"q4_k": dfx.TYPE_Q4_K, "q6_k": dfx.TYPE_Q6_K, "q8_0": dfx.TYPE_Q8_0, "f16": dfx.TYPE_F16}
ROW_BYTES = {"q4_k": 144, "q6_k": 224, "q8_0": 272, "f16": 512}     # device bytes per 256 weights
SMALL = dict(n_vocab=1536, n_embd=512, n_head=4, n_head_kv=4, n_layer=6, n_ff=1024, rope_theta=500000.0,
             rms_norm_eps=1e-5, mask_token_id=1500, is_dream=0)
SMALL_GQA = dict(n_vocab=1280, n_embd=512, n_head=8, n_head_kv=2, n_layer=3, n_ff=768, rope_theta=1000000.0,
                 rms_norm_eps=1e-6, mask_token_id=1270, is_dream=1)
SMALL_ARCH = {"small": SMALL, "small-gqa": SMALL_GQA}
DEV = "cuda"


def listed():
    return [
        # one token of ar_generate: the FFN of a decoding step (76 + 38 MB of weights, one row)
        {"name": "decode_mlp_q4k", "kind": "mlp", "arch": "dream-7b", "type": "q4_k", "M": 1},
        # the same token's attention: GQA, causal, prompt 64 + 128 tokens generated
        {"name": "decode_attn_q4k", "kind": "attn", "arch": "dream-7b", "type": "q4_k", "M": 1, "keys": 192,
         "causal": True},
        # a late cached step of a Dream-7B denoising loop (24 active rows of 128 positions)
        {"name": "step_mlp_q4k_24", "kind": "mlp", "arch": "dream-7b", "type": "q4_k", "M": 24},
        # the last cached step of the headline generation (50 active rows over 288 positions)
        {"name": "step_attn_q4k_50", "kind": "attn", "arch": "llada-8b", "type": "q4_k", "M": 50, "keys": 288,
         "causal": False},
        # an early cached step of the headline generation
        {"name": "step_mlp_q4k_245", "kind": "mlp", "arch": "llada-8b", "type": "q4_k", "M": 245},
        # its full step 0: every position is active
        {"name": "full_attn_q4k_288", "kind": "attn", "arch": "llada-8b", "type": "q4_k", "M": 288, "keys": 288,
         "causal": False},
        # the long-context unit (512 + 256 positions) on F16 weights, step 0
        {"name": "unit_mlp_f16_768", "kind": "mlp", "arch": "llada-8b", "type": "f16", "M": 768},
        # the same unit on Q8_0 weights
        {"name": "unit_attn_q8_768", "kind": "attn", "arch": "llada-8b", "type": "q8_0", "M": 768, "keys": 768,
         "causal": False},
        # a chunk of a long autoregressive prefill, up to the default context length
        {"name": "prefill_attn_q4k_4096", "kind": "attn", "arch": "dream-7b", "type": "q4_k", "M": 512, "keys": 4096,
         "causal": True},
        # the end of a cached step: vocab head over the masked rows, statistics, selection
        {"name": "step_head_q6k_74", "kind": "head", "arch": "llada-8b", "type": "q6_k", "M": 74, "policy": 2},
        # the sampler over a full block of 256 masked positions
        {"name": "sampler_256", "kind": "sampler", "arch": "llada-8b", "M": 256, "policy": 2},
        # a small model's full and cached pass through the C form of the public API: launches and host work
        {"name": "model_small", "kind": "model", "arch": "small", "scheme": "q4_k_m", "mode": "denoise", "n": 96,
         "active": 37},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: any kind, rows 1..512 (768 on the unit's types), keys up to 4096."""
    kind = rng.choice(["mlp", "mlp", "mlp", "attn", "attn", "attn", "head", "sampler", "model"])
    arch = rng.choice(["llada-8b", "dream-7b"])
    typ = rng.choice(["q4_k", "q4_k", "q4_k", "q4_k", "q8_0", "f16", "q6_k"])
    if kind in ("mlp", "attn"):
        M = _log(rng, 1, 768 if typ in ("q8_0", "f16") and arch == "llada-8b" else 512)
        c = {"kind": kind, "arch": arch, "type": typ, "M": M}
        if kind == "attn":
            c["causal"] = rng.random() < 0.4
            c["keys"] = max(M, _log(rng, max(M, 16), 4096 if M <= 256 else 2048))
        return c
    if kind == "head":
        return {"kind": kind, "arch": arch, "type": rng.choice(["q6_k", "q6_k", "q8_0", "f16"]),
                "M": _log(rng, 1, 128), "policy": rng.choice([0, 2, 4])}
    if kind == "sampler":
        return {"kind": kind, "arch": arch, "M": _log(rng, 1, 512), "policy": rng.choice([0, 2, 3, 4])}
    n = rng.randint(5, 200)
    return {"kind": "model", "arch": rng.choice(["small", "small-gqa"]),
            "scheme": rng.choice(["q4_k_m", "q8_0", "f16"]), "mode": rng.choice(["denoise", "ar"]), "n": n,
            "active": rng.randint(1, n)}


# ---------------------------------------------------------------------------
# weights: encoders into the device layout, and their decoders in 64 bits
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _f16_bytes(x):
    return x.to(torch.float16).contiguous().view(torch.uint8).reshape(*x.shape, 2)


def _encode_q4_k(w):
    n, k = w.shape
    b = w.view(n, k // 256, 8, 32)
    lo, hi = b.amin(3).clamp(max=0.0), b.amax(3)
    step, low = (hi - lo) / 15.0, -lo                                     # [n][sb][8]
    d = (step.amax(2) / 63.0).half()
    dmin = (low.amax(2) / 63.0).half()
    df, mf = d.float().unsqueeze(2), dmin.float().unsqueeze(2)
    sc = (step / df.clamp(min=1e-30)).round().clamp(0, 63)
    mn = (low / mf.clamp(min=1e-30)).round().clamp(0, 63)
    s = (df * sc).unsqueeze(3)
    q = ((b + (mf * mn).unsqueeze(3)) / s.clamp(min=1e-30)).round().clamp(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    out = torch.empty(n, k // 256, 144, dtype=torch.uint8, device=w.device)
    out[..., 0:2], out[..., 2:4] = _f16_bytes(d), _f16_bytes(dmin)
    out[..., 4:8] = sc[..., :4] | ((sc[..., 4:] >> 4) << 6)
    out[..., 8:12] = mn[..., :4] | ((mn[..., 4:] >> 4) << 6)
    out[..., 12:16] = (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)
    out[..., 16:] = (q[:, :, 0::2] | (q[:, :, 1::2] << 4)).reshape(n, k // 256, 128)
    return out.reshape(n, -1)


def _half_at(b, i):
    return b[..., i:i + 2].contiguous().view(torch.float16).double()


def _decode_q4_k(raw):
    b = raw.reshape(raw.shape[0], -1, 144)
    d, dmin = _half_at(b, 0), _half_at(b, 2)                              # [n][sb][1]
    sc = torch.cat([b[..., 4:8] & 63, (b[..., 12:16] & 15) | ((b[..., 4:8] >> 6) << 4)], 2).double()
    mn = torch.cat([b[..., 8:12] & 63, (b[..., 12:16] >> 4) | ((b[..., 8:12] >> 6) << 4)], 2).double()
    q = b[..., 16:].reshape(b.shape[0], b.shape[1], 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 3).reshape(b.shape[0], b.shape[1], 8, 32).double()
    return ((d * sc).unsqueeze(3) * q - (dmin * mn).unsqueeze(3)).reshape(b.shape[0], -1)


def _encode_q6_k(w):
    n, k = w.shape
    b = w.view(n, k // 256, 16, 16)
    a = b.abs().amax(3) / 31.0
    d = (a.amax(2) / 127.0).half()
    sc = (a / d.float().unsqueeze(2).clamp(min=1e-30)).round().clamp(0, 127)
    s = (d.float().unsqueeze(2) * sc).unsqueeze(3).clamp(min=1e-30)
    q = ((b / s).round().clamp(-32, 31) + 32).to(torch.uint8).view(n, k // 256, 2, 4, 32)
    lo = q & 15
    out = torch.zeros(n, k // 256, 224, dtype=torch.uint8, device=w.device)
    ql = torch.stack([lo[:, :, :, 0] | (lo[:, :, :, 2] << 4), lo[:, :, :, 1] | (lo[:, :, :, 3] << 4)], 3)
    h = q >> 4
    out[..., :128] = ql.reshape(n, k // 256, 128)
    out[..., 128:192] = (h[:, :, :, 0] | (h[:, :, :, 1] << 2) | (h[:, :, :, 2] << 4) |
                         (h[:, :, :, 3] << 6)).reshape(n, k // 256, 64)
    out[..., 192:208] = sc.to(torch.int8).view(torch.uint8)
    out[..., 208:210] = _f16_bytes(d)
    return out.reshape(n, -1)


def _decode_q6_k(raw, stride=224):
    b = raw.reshape(raw.shape[0], -1, stride)
    n, nsb = b.shape[:2]
    ql = b[..., :128].reshape(n, nsb, 2, 2, 32)
    qh = b[..., 128:192].reshape(n, nsb, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], 3)                                 # quarters 0, 1, 2, 3
    hi = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], 3)
    q = (lo.int() + 16 * hi.int() - 32).double().reshape(n, nsb, 16, 16)
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    return ((_half_at(b, 208) * sc).unsqueeze(3) * q).reshape(n, -1)


def _encode_q8_0(w):
    n, k = w.shape
    b = w.view(n, k // 256, 8, 32)
    d = (b.abs().amax(3) / 127.0).half()
    q = (b / d.float().unsqueeze(3).clamp(min=1e-30)).round().clamp(-127, 127).to(torch.int8)
    out = torch.empty(n, k // 256, 272, dtype=torch.uint8, device=w.device)
    out[..., :16] = _f16_bytes(d).reshape(n, k // 256, 16)
    out[..., 16:] = q.view(torch.uint8).reshape(n, k // 256, 256)
    return out.reshape(n, -1)


def _decode_q8_0(raw):
    b = raw.reshape(raw.shape[0], -1, 272)
    d = b[..., :16].contiguous().view(torch.float16).double()
    q = b[..., 16:].contiguous().view(torch.int8).double().reshape(*b.shape[:2], 8, 32)
    return (d.unsqueeze(3) * q).reshape(b.shape[0], -1)


ENCODE = {"q4_k": _encode_q4_k, "q6_k": _encode_q6_k, "q8_0": _encode_q8_0,
          "f16": lambda w: w.half().contiguous().view(torch.uint8)}
DECODE = {"q4_k": _decode_q4_k, "q6_k": _decode_q6_k, "q8_0": _decode_q8_0,
          "f16": lambda raw: raw.contiguous().view(torch.float16).double()}


def _weights(g, typ, n, k):
    """Random weights [n][k] in the device layout (encoded a few thousand rows at a time)."""
    out = torch.empty(n, k // 256 * ROW_BYTES[typ], dtype=torch.uint8, device=DEV)
    for r in range(0, n, 8192):
        m = min(8192, n - r)
        out[r:r + m] = ENCODE[typ](_randn(g, m, k) * 0.02)
    return out


def _matmul64(typ, raw, x):
    """x [M][K] (64 bits) against the decoded weights, a few thousand rows at a time."""
    out = torch.empty(x.shape[0], raw.shape[0], dtype=torch.float64, device=x.device)
    for r in range(0, raw.shape[0], 16384):
        out[:, r:r + 16384] = x @ DECODE[typ](raw[r:r + 16384]).t().contiguous()
    return out


def _activation(typ, x):
    """The activation conversion that belongs to the weight type (GGML's vec_dot_type): int8 per
    256 (Q8_K) or per 32 (Q8_0, scale in f16), or f16; the values, in 64 bits."""
    m, k = x.shape
    if typ == "f16":
        return x.float().half().double()
    if typ == "q8_0":
        b = x.view(m, k // 32, 32)
        d = b.abs().amax(2, keepdim=True) / 127.0
        q = (b / d.clamp(min=1e-300)).round()
        return (q * d.float().half().double()).view(m, k)
    b = x.view(m, k // 256, 256)
    top = b.gather(2, b.abs().argmax(2, keepdim=True))
    scale = torch.where(top == 0, torch.zeros_like(top), -127.0 / torch.where(top == 0, torch.ones_like(top), top))
    q = (b * scale).round().clamp(max=127)
    return torch.where(scale == 0, torch.zeros_like(b), q / torch.where(scale == 0, torch.ones_like(scale), scale)).view(m, k)


def _rms64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(1, keepdim=True) + eps) * w


def _stream(g, M, d):
    """A residual stream: N(0, 1) with a per-channel spread and a few large channels."""
    s = torch.exp(0.4 * _randn(g, d))
    s[torch.randint(0, d, (8,), generator=g, device=DEV)] *= 8.0
    return (_randn(g, M, d) * s).contiguous()


def _norm_weight(g, d):
    return (1.0 + 0.1 * _randn(g, d)).contiguous()


def _bytes(n):
    return torch.empty(max(int(n), 1), dtype=torch.uint8, device=DEV)


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device=DEV)


# ---------------------------------------------------------------------------
# the kinds
# ---------------------------------------------------------------------------
def _mlp_inputs(c, seed):
    a, g = ARCH[c["arch"]], _gen(seed)
    d, F = a["n_embd"], a["n_ff"]
    return dict(x=_stream(g, c["M"], d), norm=_norm_weight(g, d), gu=_weights(g, c["type"], 2 * F, d),
                down=_weights(g, c["type"], d, F))


def _mlp_prepare(c, seed):
    a, t, M = ARCH[c["arch"]], TYPE[c["type"]], c["M"]
    d, F, L = a["n_embd"], a["n_ff"], dfx.lib()
    i = _mlp_inputs(c, seed)
    act = _bytes(max(L.dfx_act_bytes(t, M, d), L.dfx_act_bytes(t, M, F)))
    ws = _bytes(max(L.dfx_gemm_ws_bytes(M, 2 * F, d), L.dfx_gemm_ws_bytes(M, d, F)))
    h, y = _f32(M, F), _f32(M, d)
    x, A, W = i["x"].data_ptr(), act.data_ptr(), ws.data_ptr()
    calls = [
        (L.dfx_rmsnorm_convert, (t, x, i["norm"].data_ptr(), M, d, a["rms_norm_eps"], A, None)),
        (L.dfx_gemm_swiglu, (t, i["gu"].data_ptr(), 2 * F, d, A, M, h.data_ptr(), F, W, None)),
        (L.dfx_act_convert, (t, h.data_ptr(), M, F, A, None)),
        (L.dfx_gemm, (t, i["down"].data_ptr(), d, F, A, M, None, x, y.data_ptr(), W, None)),
    ]
    return dict(calls=calls, out=y, keep=(i, act, ws, h))


def _mlp_exact(c, seed):
    a, t = ARCH[c["arch"]], c["type"]
    i = _mlp_inputs(c, seed)
    x = i["x"].double()
    z = _matmul64(t, i["gu"], _activation(t, _rms64(x, i["norm"].double(), a["rms_norm_eps"])))
    z = z.view(c["M"], -1, 2, 16)                       # rows: 16 of gate, 16 of up, alternating
    gate, up = z[:, :, 0].reshape(c["M"], -1), z[:, :, 1].reshape(c["M"], -1)
    return _matmul64(t, i["down"], _activation(t, torch.nn.functional.silu(gate) * up)) + x


def _mlp_work(c):
    a, M, rb = ARCH[c["arch"]], c["M"], ROW_BYTES[c["type"]]
    d, F = a["n_embd"], a["n_ff"]
    return {"bytes": 3 * d * F // 256 * rb + 8 * M * d + 4 * d, "flops": 2.0 * M * 3 * d * F}


def _attn_dims(c):
    a = ARCH[c["arch"]]
    H, Hkv = a["n_head"], a["n_head_kv"]
    return a["n_embd"], H, Hkv, a["n_embd"] // H, (c["keys"] + 15) // 16 * 16


def _attn_inputs(c, seed):
    a, g, M, keys = ARCH[c["arch"]], _gen(seed), c["M"], c["keys"]
    d, H, Hkv, hd, cap = _attn_dims(c)
    n = (H + 2 * Hkv) * hd
    i = dict(x=_stream(g, M, d), norm=_norm_weight(g, d), qkv=_weights(g, c["type"], n, d),
             o=_weights(g, c["type"], d, d), bias=0.1 * _randn(g, n) if a["is_dream"] else None,
             kc=1.2 * _randn(g, cap, Hkv * hd), vt=1.2 * _randn(g, Hkv, hd, cap))
    if c["causal"]:
        i["pos"] = torch.arange(keys - M, keys, device=DEV, dtype=torch.int32)
    else:
        i["pos"] = torch.randperm(keys, generator=g, device=DEV)[:M].sort().values.to(torch.int32)
    ang = torch.arange(cap, device=DEV, dtype=torch.float64)[:, None] * torch.pow(
        torch.tensor(a["rope_theta"], dtype=torch.float64, device=DEV),
        -torch.arange(hd // 2, device=DEV, dtype=torch.float64) * 2.0 / hd)
    i["tab"] = torch.stack([ang.cos(), ang.sin()], 2).float().contiguous()
    return i


def _attn_prepare(c, seed):
    a, t, M, keys = ARCH[c["arch"]], TYPE[c["type"]], c["M"], c["keys"]
    d, H, Hkv, hd, cap = _attn_dims(c)
    n, L = (H + 2 * Hkv) * hd, dfx.lib()
    i = _attn_inputs(c, seed)
    act = _bytes(L.dfx_act_bytes(t, M, d))
    ws = _bytes(max(L.dfx_gemm_ws_bytes(M, n, d), L.dfx_gemm_ws_bytes(M, d, d)))
    q, att, y = _f32(M, H, hd), _f32(M, d), _f32(M, d)
    x, A, W, KC, VT = (v.data_ptr() for v in (i["x"], act, ws, i["kc"], i["vt"]))
    bias = i["bias"].data_ptr() if i["bias"] is not None else None
    if c["causal"]:
        attend = (L.dfx_attention_causal, (q.data_ptr(), KC, VT, cap, M, keys, H, Hkv, hd, keys - M, 0, att.data_ptr(),
                                           None))
    else:
        attend = (L.dfx_attention, (q.data_ptr(), KC, VT, cap, M, keys, H, Hkv, hd, att.data_ptr(), None))
    calls = [
        (L.dfx_rmsnorm_convert, (t, x, i["norm"].data_ptr(), M, d, a["rms_norm_eps"], A, None)),
        (L.dfx_gemm_rope, (t, i["qkv"].data_ptr(), n, d, A, M, bias, 0, i["pos"].data_ptr(), H, Hkv, hd,
                           i["tab"].data_ptr(), q.data_ptr(), KC, VT, cap, W, None)),
        attend,
        (L.dfx_act_convert, (t, att.data_ptr(), M, d, A, None)),
        (L.dfx_gemm, (t, i["o"].data_ptr(), d, d, A, M, None, x, y.data_ptr(), W, None)),
    ]
    return dict(calls=calls, out={"y": y, "kc": i["kc"], "vt": i["vt"]}, keep=(i, act, ws, q, att))


def _rope64(v, tab, pos):
    """v [M][heads][hd] in natural order, rotated in NEOX pairs (i, i + hd/2)."""
    cs = tab[pos.long()].double()
    c, s, h = cs[:, None, :, 0], cs[:, None, :, 1], v.shape[2] // 2
    a, b = v[..., :h], v[..., h:]
    return torch.cat([a * c - b * s, a * s + b * c], 2)


def _attend64(q, k, v, q_pos, causal):
    """q [M][H][hd], k / v [keys][Hkv][hd] -> [M][H * hd]; one head at a time."""
    M, H, hd = q.shape
    out = torch.empty(M, H, hd, dtype=torch.float64, device=q.device)
    hide = torch.arange(k.shape[0], device=q.device)[None, :] > q_pos[:, None] if causal else None
    for h in range(H):
        kv = h // (H // k.shape[1])
        s = q[:, h] @ k[:, kv].t().contiguous() / math.sqrt(hd)
        if causal:
            s = s.masked_fill(hide, -math.inf)
        out[:, h] = torch.softmax(s, 1) @ v[:, kv].contiguous()
    return out.reshape(M, H * hd)


def _attn_exact(c, seed):
    a, t, M, keys = ARCH[c["arch"]], c["type"], c["M"], c["keys"]
    d, H, Hkv, hd, cap = _attn_dims(c)
    i = _attn_inputs(c, seed)
    x = i["x"].double()
    z = _matmul64(t, i["qkv"], _activation(t, _rms64(x, i["norm"].double(), a["rms_norm_eps"])))
    if i["bias"] is not None:
        z = z + i["bias"].double()
    z = z.view(M, H + 2 * Hkv, hd)
    # Q and K rows: blocks of 32 hold dims 16j.. then the dims hd/2 + 16j.. they rotate with
    qk = z[:, :H + Hkv].reshape(M, H + Hkv, hd // 32, 2, 16).transpose(2, 3).reshape(M, H + Hkv, hd)
    qk = _rope64(qk, i["tab"], i["pos"])
    kc, vt, p = i["kc"].double(), i["vt"].double(), i["pos"].long()
    kc[p] = qk[:, H:].reshape(M, -1)
    vt[:, :, p] = z[:, H + Hkv:].permute(1, 2, 0)
    att = _attend64(qk[:, :H], kc[:keys].view(keys, Hkv, hd), vt[:, :, :keys].permute(2, 0, 1), p, c["causal"])
    return {"y": _matmul64(t, i["o"], _activation(t, att)) + x, "kc": kc, "vt": vt}


def _attn_work(c):
    d, H, Hkv, hd, cap = _attn_dims(c)
    M, keys, n = c["M"], c["keys"], (H + 2 * Hkv) * hd
    seen = M * keys - M * (M - 1) / 2 if c["causal"] else M * keys
    return {"bytes": (n + d) * d // 256 * ROW_BYTES[c["type"]] + 8 * keys * Hkv * hd + 8 * M * d + 8 * M * Hkv * hd,
            "flops": 2.0 * M * (n + d) * d + 4.0 * seen * H * hd}


def _head_inputs(c, seed):
    a, g, M = ARCH[c["arch"]], _gen(seed), c["M"]
    d, V = a["n_embd"], a["n_vocab"]
    w = _weights(g, c["type"], V, d)
    # rows that lean towards one token each, from not at all to clearly, as in mid-generation
    tok = torch.randint(0, V, (M,), generator=g, device=DEV)
    dir_ = DECODE[c["type"]](w[tok]).float()
    lean = 0.3 * torch.rand(M, 1, generator=g, device=DEV)
    x = _randn(g, M, d) + lean * math.sqrt(d) * dir_ / dir_.norm(dim=1, keepdim=True)
    return dict(x=x.contiguous(), norm=torch.ones(d, device=DEV), w=w)


def _sampler_buffers(M):
    stats = torch.empty(M, 4, dtype=torch.int32, device=DEV)
    cand = torch.empty(M, 4, dtype=torch.int32, device=DEV)
    order = torch.empty(M, dtype=torch.int32, device=DEV)
    nun = torch.empty(1, dtype=torch.int32, device=DEV)
    rows = torch.arange(M, dtype=torch.int32, device=DEV)
    pos = 32 + 2 * rows
    return dict(stats=stats, cand=cand, order=order, nun=nun, rows=rows, pos=pos)


def _sampler_calls(L, c, logits, b):
    V, M = ARCH[c["arch"]]["n_vocab"], c["M"]
    p = {k: v.data_ptr() for k, v in b.items()}
    return [(L.dfx_row_stats, (logits.data_ptr(), V, p["rows"], M, V, p["stats"], None)),
            (L.dfx_select_from_stats, (p["stats"], p["pos"], M, c["policy"], 1.5, max(1, M // 8), p["cand"],
                                       p["order"], p["nun"], None))]


def _sampler_out(b):
    s, k = b["stats"], b["cand"]
    return {"token": s[:, 0], "stat": s.view(torch.float32)[:, 1:], "cand": k[:, :2],
            "key": k.view(torch.float32)[:, 2:], "order": b["order"], "n": b["nun"]}


def _head_prepare(c, seed):
    a, t, M, L = ARCH[c["arch"]], TYPE[c["type"]], c["M"], dfx.lib()
    d, V = a["n_embd"], a["n_vocab"]
    i = _head_inputs(c, seed)
    act, logits, b = _bytes(L.dfx_act_bytes(t, M, d)), _f32(M, V), _sampler_buffers(M)
    calls = [(L.dfx_rmsnorm_convert, (t, i["x"].data_ptr(), i["norm"].data_ptr(), M, d, a["rms_norm_eps"],
                                      act.data_ptr(), None)),
             (L.dfx_gemm, (t, i["w"].data_ptr(), V, d, act.data_ptr(), M, None, None, logits.data_ptr(), None, None))]
    return dict(calls=calls + _sampler_calls(L, c, logits, b), out=dict(_sampler_out(b), logits=logits),
                keep=(i, act, b))


def _stats64(c, logits):
    p = torch.log_softmax(logits, 1)
    top = logits.topk(2, 1).values
    ent = -(p.exp() * p).sum(1)
    stat = torch.cat([top, ent[:, None]], 1)
    conf = top[:, 0] - top[:, 1] if c["policy"] == dfx.TOPK_MARGIN else top[:, 0]
    return {"token": None, "stat": stat, "cand": None, "key": torch.stack([conf, ent], 1), "order": None, "n": None}


def _head_exact(c, seed):
    a, t = ARCH[c["arch"]], c["type"]
    i = _head_inputs(c, seed)
    logits = _matmul64(t, i["w"], _activation(t, _rms64(i["x"].double(), i["norm"].double(), a["rms_norm_eps"])))
    return dict(_stats64(c, logits), logits=logits)


def _head_work(c):
    a, M = ARCH[c["arch"]], c["M"]
    d, V = a["n_embd"], a["n_vocab"]
    return {"bytes": V * d // 256 * ROW_BYTES[c["type"]] + 4 * M * V + 4 * M * d, "flops": 2.0 * M * V * d}


def _sampler_logits(c, seed):
    g, M, V = _gen(seed), c["M"], ARCH[c["arch"]]["n_vocab"]
    # from near-uniform rows (entropy about 11) to rows that a few tokens dominate
    scale = 0.5 + 5.5 * torch.rand(M, 1, generator=g, device=DEV)
    return (_randn(g, M, V) * scale).contiguous()


def _sampler_prepare(c, seed):
    logits, b = _sampler_logits(c, seed), _sampler_buffers(c["M"])
    return dict(calls=_sampler_calls(dfx.lib(), c, logits, b), out=_sampler_out(b), keep=(logits, b))


def _sampler_exact(c, seed):
    return _stats64(c, _sampler_logits(c, seed).double())


def _sampler_work(c):
    V = ARCH[c["arch"]]["n_vocab"]
    return {"bytes": 4 * c["M"] * V + 52 * c["M"], "flops": 6.0 * c["M"] * V}


# ---- whole passes of a small model
class _File:
    """A model file, and what a program keeps of it; the file goes with the object."""

    def __init__(self, c, seed):
        fd, self.path = tempfile.mkstemp(suffix=".gguf")
        os.close(fd)
        dfx.synth_model(self.path, SMALL_ARCH[c["arch"]], scheme=c["scheme"], seed=seed, sigma=0.05, n_threads=4)

    def __del__(self):
        os.unlink(self.path)


def _model_inputs(c, seed):
    r = np.random.default_rng(seed)
    V, n = SMALL_ARCH[c["arch"]]["n_vocab"], c["n"]
    return dict(tokens=r.integers(0, V, n).astype(np.int32),
                pos=np.sort(r.permutation(n)[:c["active"]]).astype(np.int32),
                fresh=r.integers(0, V, c["active"] if c["mode"] == "denoise" else 4).astype(np.int32))


def _model_prepare(c, seed):
    f = _File(c, seed)
    model = dfx.Model(f.path)
    return dict(_model_inputs(c, seed), ctx=dfx.Context(model, c["n"] + 8), mode=c["mode"], keep=(f, model))


def _model_run(s):
    ctx = s["ctx"]
    if s["mode"] == "denoise":       # a full forward, then a cached step over some of its positions
        return {"full": ctx.forward(s["tokens"]), "cached": ctx.forward_cached(s["fresh"], s["pos"], len(s["tokens"]))}
    out = {"prefill": ctx.ar_forward(s["tokens"], reset=True)}
    for k in range(4):               # then four tokens, one at a time
        out["token%d" % k] = ctx.ar_forward(s["fresh"][k:k + 1])
    return out


def _gguf(path):
    """{tensor name: (type id, raw uint8 rows [n][bytes])} of a GGUF file."""
    raw = np.fromfile(path, dtype=np.uint8)
    at = [8]

    def u(fmt):
        v = struct.unpack_from("<" + fmt, raw, at[0])[0]
        at[0] += struct.calcsize(fmt)
        return v

    def text():
        n = u("Q")
        at[0] += n
        return raw[at[0] - n:at[0]].tobytes().decode()

    size = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}
    n_tensors, n_kv = u("Q"), u("Q")
    for _ in range(n_kv):
        text()
        kind = u("I")
        if kind == 8:
            text()
        else:
            at[0] += size[kind]
    infos = []
    for _ in range(n_tensors):
        name = text()
        dims = [u("Q") for _ in range(u("I"))]
        infos.append((name, dims, u("I"), u("Q")))
    base = (at[0] + 31) // 32 * 32
    geom = {0: (1, 4), 1: (1, 2), 8: (32, 34), 12: (256, 144), 14: (256, 210)}
    out = {}
    for name, dims, typ, off in infos:
        blk, nb = geom[typ]
        rows = dims[1] if len(dims) > 1 else 1
        out[name] = (typ, raw[base + off:base + off + rows * (dims[0] // blk) * nb].reshape(rows, -1))
    return out


def _tensor64(t):
    typ, raw = t
    raw = torch.from_numpy(raw.copy()).to(DEV)
    if typ == dfx.TYPE_F32:
        return raw.view(torch.float32).double()
    if typ == dfx.TYPE_F16:
        return raw.view(torch.float16).double()
    if typ == dfx.TYPE_Q8_0:
        b = raw.view(raw.shape[0], -1, 34)
        return (_half_at(b, 0) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(raw.shape[0], -1)
    return _decode_q4_k(raw) if typ == dfx.TYPE_Q4_K else _decode_q6_k(raw, 210)


def _model_exact(c, seed):
    a, i = SMALL_ARCH[c["arch"]], _model_inputs(c, seed)
    f = _File(c, seed)
    T = _gguf(f.path)
    d, H, Hkv, eps = a["n_embd"], a["n_head"], a["n_head_kv"], a["rms_norm_eps"]
    hd, causal = d // H, c["mode"] == "ar"
    conv = {dfx.TYPE_Q4_K: "q4_k", dfx.TYPE_Q6_K: "q6_k", dfx.TYPE_Q8_0: "q8_0", dfx.TYPE_F16: "f16"}
    w64 = {n: _tensor64(t) for n, t in T.items()}
    total = c["n"] + (4 if causal else 0)
    # theta_0 = p, theta_{i+1} = theta_i * base^(-2/hd) in f32, as GGML's rope cache
    th = np.zeros((total, hd // 2), np.float32)
    th[:, 0] = np.arange(total)
    step = np.float32(np.float32(a["rope_theta"]) ** np.float32(-2.0 / hd))
    for k in range(1, hd // 2):
        th[:, k] = th[:, k - 1] * step
    ang = torch.from_numpy(th).to(DEV).double()
    tab = torch.stack([ang.cos(), ang.sin()], 2)
    cache = [[torch.zeros(total, Hkv, hd, dtype=torch.float64, device=DEV) for _ in range(2)]
             for _ in range(a["n_layer"])]

    def mul(name, x):
        y = _activation(conv[T[name + ".weight"][0]], x) @ w64[name + ".weight"].t().contiguous()
        return y + w64[name + ".bias"].reshape(-1) if name + ".bias" in w64 else y

    def norm(name, x):
        return _rms64(x, w64[name + ".weight"].reshape(-1), eps)

    def forward(tokens, pos, keys):
        p = torch.as_tensor(pos, device=DEV).long()
        x = w64["token_embd.weight"][torch.as_tensor(tokens, device=DEV).long()]
        for il in range(a["n_layer"]):
            b, m = "blk.%d." % il, len(pos)
            z = norm(b + "attn_norm", x)
            q = _rope64(mul(b + "attn_q", z).view(m, H, hd), tab, p)
            cache[il][0][p] = _rope64(mul(b + "attn_k", z).view(m, Hkv, hd), tab, p)
            cache[il][1][p] = mul(b + "attn_v", z).view(m, Hkv, hd)
            x = x + mul(b + "attn_output", _attend64(q, cache[il][0][:keys], cache[il][1][:keys], p, causal))
            z = norm(b + "ffn_norm", x)
            x = x + mul(b + "ffn_down", torch.nn.functional.silu(mul(b + "ffn_gate", z)) * mul(b + "ffn_up", z))
        return mul("output", norm("output_norm", x)).cpu().numpy()

    n = c["n"]
    if not causal:
        return {"full": forward(i["tokens"], np.arange(n), n), "cached": forward(i["fresh"], i["pos"], n)}
    out = {"prefill": forward(i["tokens"], np.arange(n), n)}
    for k in range(4):
        out["token%d" % k] = forward(i["fresh"][k:k + 1], np.array([n + k]), n + k + 1)
    return out


def _model_work(c):
    a = SMALL_ARCH[c["arch"]]
    d, F, L, V = a["n_embd"], a["n_ff"], a["n_layer"], a["n_vocab"]
    dkv = d // a["n_head"] * a["n_head_kv"]
    per = L * (2 * d * d + 2 * d * dkv + 3 * d * F) + V * d
    rows = [c["n"], c["active"]] if c["mode"] == "denoise" else [c["n"], 1, 1, 1, 1]
    width = {"q4_k_m": 0.6, "q8_0": 1.07, "f16": 2.0}[c["scheme"]]
    return {"bytes": sum(per * width + 4 * r * V for r in rows),
            "flops": sum(2.0 * per * r + 4.0 * r * c["n"] * d * L for r in rows)}


# ---------------------------------------------------------------------------
PREPARE = {"mlp": _mlp_prepare, "attn": _attn_prepare, "head": _head_prepare, "sampler": _sampler_prepare,
           "model": _model_prepare}
EXACT = {"mlp": _mlp_exact, "attn": _attn_exact, "head": _head_exact, "sampler": _sampler_exact,
         "model": _model_exact}
WORK = {"mlp": _mlp_work, "attn": _attn_work, "head": _head_work, "sampler": _sampler_work, "model": _model_work}


def prepare(case, seed):
    return PREPARE[case["kind"]](case, seed)


def run(state):
    if "ctx" in state:
        return _model_run(state)
    for fn, args in state["calls"]:
        dfx.check(fn(*args))
    return state["out"]


def exact(case, seed):
    with torch.no_grad():
        return EXACT[case["kind"]](case, seed)


def work(case):
    return WORK[case["kind"]](case)


def tolerance(case):
    """Every GEMM re-quantises its input (int8 per 256 or 32, or f16), so a float sum in another
    order moves a few inputs of the next GEMM by a whole quantisation step.  Measured against
    exact(): blocks on quantised weights 1e-4..5e-4, the head 3e-5, F16 blocks 3e-5, the sampler
    2e-8 (f32 results of f64 or f32 sums), the small model 0.05 after six layers of such steps
    (of which 0.03 is the most that is allowed); about four times that is allowed."""
    if case["kind"] == "sampler":
        return {"rel": 1e-6, "max": 1e-4, "differ": 0.01}
    if case["kind"] == "model":
        return {"rel": 0.03, "max": 0.5}
    if case["type"] == "f16":
        return {"rel": 2e-4, "max": 0.02, "differ": 0.01}
    if case["kind"] == "head":
        return {"rel": 2e-4, "max": 0.02, "differ": 0.01}
    return {"rel": 2e-3, "max": 0.08, "differ": 0.01}
