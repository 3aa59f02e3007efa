"""What the speed of this framework is measured on.

The framework runs llama / qwen2 / qwen3 / qwen3moe GGUF models: a decode step is a chain of one-token
matvecs over quantised weights with an attention over the cached positions, a prompt is the same chain
over up to a few hundred tokens at a time. The cases are those layers, each through the entry point the
engine calls for it (the C ABI bound in sardyne_amd.capi), and two whole evaluations through
sardyne_amd.engine:

- "linear": one weight matrix times n_tok activation rows, quantised (after an RMSNorm where the layer
  has one) as the weight's format asks: projections, gate|up with SwiGLU, down, the output head;
- "prompt_attention" / "decode_attention": causal attention of a prompt chunk over the cache, and the
  one-token attention with its q/k norm, RoPE and cache write;
- "engine": a few layers of a whole model, decoding some tokens or evaluating a prompt.

Weights are random blocks in the GGUF formats with the scale structure of model files (the largest
sub-block scale of a super-block at the end of its range) and a standard deviation of 1/sqrt(n_in).
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

from sardyne_amd import capi
from sardyne_amd.engine import LoadedModel
from sardyne_amd.gguf_synth import GGUFBuilder

DEV = "cuda"
EPS = 1e-6
# GGUF type ids; elements and bytes of a block
TYPES = {"F32": (0, 1, 4), "F16": (1, 1, 2), "Q4_0": (2, 32, 18), "Q5_0": (6, 32, 22), "Q8_0": (8, 32, 34),
         "Q4_K": (12, 256, 144), "Q6_K": (14, 256, 210), "BF16": (30, 1, 2)}
FLOAT = ("F32", "F16", "BF16")
K_QUANT = ("Q4_K", "Q6_K")
Q8_0, Q8_K = 8, 15
MAX_SEQ_PAD = 64  # positions a cache has beyond the ones a case fills


# ------------------------------------------------------------------------------------------ cases

def listed():
    return [
        # attention output projection of one decoded token: the smallest call of a step
        _linear("proj_q4k_1", "Q4_K", 2048, 2048, 1, resid=True),
        # the output head of a decode step (final norm included): a quarter GB read per token
        _linear("head_q6k_1", "Q6_K", 2048, 151936, 1, norm=True),
        # logits of every position of a 64-token batch (scoring a text)
        _linear("head_q6k_64", "Q6_K", 2048, 151936, 64, norm=True),
        # the FFN's gate|up for a short user turn
        _linear("gate_up_q4k_7", "Q4_K", 2048, 22016, 7, norm=True, swiglu=True),
        # the same for a full prompt chunk
        _linear("gate_up_q4k_512", "Q4_K", 2048, 22016, 512, norm=True, swiglu=True),
        # the FFN's down for a prompt of some ragged length
        _linear("down_q6k_203", "Q6_K", 11008, 2048, 203, resid=True),
        # a prompt chunk through an 8-bit file
        _linear("gate_up_q8_0_512", "Q8_0", 2048, 22016, 512, norm=True, swiglu=True),
        # a half-precision file's projection over a prompt
        _linear("proj_f16_128", "F16", 2048, 2048, 128),
        # a prompt's third 512-token chunk
        {"name": "attn_prompt_512", "kind": "prompt_attention", "n_tok": 512, "past": 1024, "n_head": 32,
         "n_kv_head": 4, "head_dim": 128, "kv": "f32"},
        # one token at the end of a long conversation
        {"name": "attn_decode_9001", "kind": "decode_attention", "past": 9001, "n_head": 16, "n_kv_head": 2,
         "head_dim": 128, "kv": "f16", "qk_norm": False},
        # chat: tokens decoded one after another
        {"name": "engine_decode", "kind": "engine", "arch": "qwen2", "file": "Q4_K_M", "n_layer": 2, "vocab": 32000,
         "past": 513, "n_tok": 4, "decode": True},
        # a prompt through a mixture-of-experts layer
        {"name": "engine_prompt_moe", "kind": "engine", "arch": "qwen3moe", "file": "Q4_K_M", "n_layer": 1,
         "vocab": 32000, "past": 0, "n_tok": 301, "decode": False},
    ]


def _linear(name, wtype, n_in, n_out, n_tok, norm=False, swiglu=False, resid=False):
    return {"name": name, "kind": "linear", "wtype": wtype, "n_in": n_in, "n_out": n_out, "n_tok": n_tok,
            "norm": norm, "swiglu": swiglu, "resid": resid}


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["prompt_attention", "decode_attention", "engine", "engine"])
    if kind == "linear":
        wtype = rng.choice(["Q4_K"] * 4 + ["Q6_K"] * 3 + ["Q8_0"] * 3 + ["Q4_0", "Q5_0", "F16", "BF16", "F32"])
        block = 256 if wtype in K_QUANT else 32 if wtype not in FLOAT else 4
        n_in = block * _log_int(rng, -(-512 // block), 11008 // block)
        n_tok = rng.choice([1, _log_int(rng, 2, 15), _log_int(rng, 16, 512)])
        most = 151936 * 2048 if wtype not in FLOAT else 2048 * 8192
        most = min(most // n_in, 22016 * 2048 * 512 // (n_in * n_tok), 151936)
        if wtype in FLOAT:
            most = min(most, 2048 * 2048 * 256 // (n_in * n_tok))
        n_out = _log_int(rng, 97, most)
        swiglu = wtype not in FLOAT and rng.random() < 0.3
        if swiglu:
            n_out += n_out % 2
        norm = rng.random() < 0.5
        return {"kind": "linear", "wtype": wtype, "n_in": n_in, "n_out": n_out, "n_tok": n_tok, "norm": norm,
                "swiglu": swiglu, "resid": not norm and not swiglu and rng.random() < 0.5}
    n_kv_head = rng.choice([1, 2, 4, 8])
    n_head = n_kv_head * rng.choice([1, 2, 4, 8] if n_kv_head < 8 else [1, 2, 4])
    if kind == "prompt_attention":
        return {"kind": kind, "n_tok": _log_int(rng, 2, 512), "past": _log_int(rng, 1, 1024), "n_head": n_head,
                "n_kv_head": n_kv_head, "head_dim": rng.choice([64, 128]), "kv": rng.choice(["f32", "f16"])}
    if kind == "decode_attention":
        return {"kind": kind, "past": _log_int(rng, 16, 16384), "n_head": n_head, "n_kv_head": n_kv_head,
                "head_dim": rng.choice([64, 128]), "kv": rng.choice(["f32", "f16"]),
                "qk_norm": rng.random() < 0.5}
    moe = rng.random() < 0.4
    decode = rng.random() < 0.5
    return {"kind": "engine", "arch": "qwen3moe" if moe else "qwen2",
            "file": "Q4_K_M" if moe else rng.choice(["Q4_K_M", "Q8_0"]), "n_layer": 1,
            "vocab": rng.choice([32000, 16001]), "past": rng.choice([0, _log_int(rng, 1, 1000)]) if not decode
            else _log_int(rng, 1, 1000), "n_tok": _log_int(rng, 1, 6) if decode else _log_int(rng, 2, 301),
            "decode": decode}


# --------------------------------------------------------------------------- weights in GGUF's formats

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device=DEV, dtype=torch.uint8)


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _spread(g, n, base):
    """n block scales around base"""
    return base * torch.empty(n, device=DEV).uniform_(0.6, 1.4, generator=g)


def _blocks(wtype, rows, n_in, g):
    """Random rows of a matrix as its GGUF bytes, [rows][row bytes], of standard deviation 1/sqrt(n_in)."""
    std = 1.0 / math.sqrt(n_in)
    if wtype in FLOAT:
        w = _randn(g, rows, n_in) * std
        return w.to({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[wtype]).view(torch.uint8)
    _, block, size = TYPES[wtype]
    n = rows * n_in // block
    b = _bytes(g, n, size)
    if wtype == "Q4_K":
        # 6-bit scales up to 63, minima that centre the 4-bit quants
        sc = torch.randint(20, 64, (n, 8), generator=g, device=DEV, dtype=torch.uint8)
        mn = torch.randint(20, 64, (n, 8), generator=g, device=DEV, dtype=torch.uint8)
        for v in (sc, mn):
            v[torch.arange(n, device=DEV), torch.randint(0, 8, (n,), generator=g, device=DEV)] = 63
        d = _spread(g, n, std / (4.6 * 44))
        b[:, 0:2] = _f16_bytes(d)
        b[:, 2:4] = _f16_bytes(7.5 * d)
        b[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        b[:, 8:12] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
        b[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    elif wtype == "Q6_K":
        # int8 scales, the largest amplitude of a super-block at -128
        sc = torch.randint(40, 128, (n, 16), generator=g, device=DEV, dtype=torch.int16)
        sc = sc * (1 - 2 * torch.randint(0, 2, (n, 16), generator=g, device=DEV, dtype=torch.int16))
        sc[torch.arange(n, device=DEV), torch.randint(0, 16, (n,), generator=g, device=DEV)] = -128
        b[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _f16_bytes(_spread(g, n, std / (18.5 * 88)))
    else:
        top = {"Q8_0": 73.0, "Q4_0": 4.6, "Q5_0": 9.2}[wtype]
        b[:, 0:2] = _f16_bytes(_spread(g, n, std / top))
    return b.reshape(rows, -1)


def _values(wtype, raw, n_in):
    """The rows of _blocks as float64 numbers, [rows][n_in]."""
    rows = raw.shape[0]
    if wtype in FLOAT:
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[wtype]
        return raw.contiguous().view(t).reshape(rows, n_in).double()
    _, block, size = TYPES[wtype]
    b = raw.reshape(-1, size)
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if wtype == "Q4_K":
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16:144].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        w = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    elif wtype == "Q6_K":
        lo, hi = b[:, 0:128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        lo = torch.cat([lo & 15, lo >> 4], 2)  # [2 halves][4 quarters][32]
        hi = torch.cat([(hi >> (2 * i)) & 3 for i in range(4)], 2)
        q = (lo | (hi << 4)).reshape(-1, 16, 16).double() - 32
        w = (half(208) * b[:, 192:208].contiguous().view(torch.int8).double())[:, :, None] * q
    elif wtype == "Q8_0":
        w = half(0) * b[:, 2:34].contiguous().view(torch.int8).double()
    elif wtype == "Q4_0":
        w = half(0) * (torch.cat([b[:, 2:18] & 15, b[:, 2:18] >> 4], 1).double() - 8)
    else:
        qh = b[:, 2:6].to(torch.int64)
        qh = qh[:, 0] | (qh[:, 1] << 8) | (qh[:, 2] << 16) | (qh[:, 3] << 24)
        bit = (qh[:, None] >> torch.arange(32, device=DEV)) & 1
        w = half(0) * ((torch.cat([b[:, 6:22] & 15, b[:, 6:22] >> 4], 1).long() | (bit << 4)).double() - 16)
    return w.reshape(rows, n_in)


def _activations(wtype, x):
    """What the weight format multiplies: the rows of x themselves, or their 8-bit blocks (the block scales
    and quotients in the 32 bits that define them: tensors divided by tensors, since torch turns a division of or by
    a number into a product with a reciprocal), as float64."""
    if wtype in FLOAT:
        return x.double()
    n = 256 if wtype in K_QUANT else 32
    v = x.float().reshape(-1, n)
    at = v.abs().argmax(1, keepdim=True)
    if wtype in K_QUANT:
        top = v.gather(1, at)
        inv = torch.where(top == 0, torch.zeros_like(top), torch.full_like(top, -127.0) / top)
        q = torch.clamp(torch.round(inv * v), max=127)
        d = torch.where(inv == 0, torch.zeros_like(inv), torch.ones_like(inv) / inv)
    else:
        d = v.abs().gather(1, at)
        d = d / torch.full_like(d, 127.0)
        inv = torch.where(d == 0, torch.zeros_like(d), torch.ones_like(d) / d)
        y = v * inv
        q = torch.sign(y) * torch.floor(y.abs() + 0.5)
        d = d.to(torch.float16)
    return (q.double() * d.double()).reshape(x.shape)


def _norm(x, w):
    scale = (1.0 / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + EPS)).float()
    return x.float() * scale * w


def _product(wtype, raw, x, n_in):
    """x . W^T in float64, in pieces of rows that fit"""
    a = _activations(wtype, x)
    step = max(1, (1 << 27) // n_in)
    return torch.cat([a @ _values(wtype, raw[r:r + step], n_in).T for r in range(0, raw.shape[0], step)], 1)


# ------------------------------------------------------------------------------------------- states

class _Matrix:
    """A weight matrix uploaded as the engine uploads one, with the prompt GEMM's copy of it."""

    def __init__(self, wtype, n_in, raw):
        self.m = capi.SdyMat()
        capi.check(capi.lib().sdy_mat_from_device(ctypes.byref(self.m), TYPES[wtype][0], n_in, raw.shape[0],
                                                  raw.data_ptr(), None))
        capi.check(capi.lib().sdy_mat_gemm_layout(ctypes.byref(self.m), None))

    def __del__(self):
        capi.lib().sdy_mat_free(ctypes.byref(self.m))


class _Calls:
    """The library calls of a pass, in order, their arguments laid out once, and the tensors they write."""

    def __init__(self, calls, out, keep):
        self.calls, self.out, self.keep = calls, out, keep


def _linear_inputs(case, seed):
    g = _gen(seed)
    raw = _blocks(case["wtype"], case["n_out"], case["n_in"], g)
    x = _randn(g, case["n_tok"], case["n_in"])
    nw = torch.empty(case["n_in"], device=DEV).uniform_(0.5, 1.5, generator=g) if case["norm"] else None
    resid = _randn(g, case["n_tok"], case["n_out"]) if case["resid"] else None
    return raw, x, nw, resid


def _prepare_linear(case, seed):
    lib = capi.lib()
    wtype, n_in, n_out, n_tok = case["wtype"], case["n_in"], case["n_out"], case["n_tok"]
    raw, x, nw, resid = _linear_inputs(case, seed)
    mat = _Matrix(wtype, n_in, raw)
    m = ctypes.byref(mat.m)
    cols = n_out // 2 if case["swiglu"] else n_out
    out = torch.zeros(n_tok, cols, device=DEV)
    a = capi.SdyMvArgs(n_tok=n_tok, out=out.data_ptr(), out_stride=cols, row0=0, row1=n_out,
                       resid=resid.data_ptr() if resid is not None else None,
                       epilogue=capi.EPI_SWIGLU if case["swiglu"] else capi.EPI_NONE, eps=EPS)
    keep, calls = [mat, x, nw, resid, a], []
    xp, nwp = x.data_ptr(), nw.data_ptr() if nw is not None else None
    arg = ctypes.byref(a)
    if wtype in FLOAT:
        a.x = xp
        if nw is not None:
            xb = torch.empty_like(x)
            keep.append(xb)
            a.x = xb.data_ptr()
            calls.append((lib.sdy_norm_quant, (xp, nwp, EPS, n_in, n_tok, xb.data_ptr(), TYPES["F32"][0], None, None)))
        calls.append((lib.sdy_matvec, (m, arg, None)))
        return _Calls(calls, out, keep)
    vt = Q8_K if wtype in K_QUANT else Q8_0
    a.x, a.nw = xp, nwp
    if n_tok == 1 and lib.sdy_matvec_fused_ok(m, arg, None, None):
        calls.append((lib.sdy_matvec, (m, arg, None)))
        return _Calls(calls, out, keep)
    a.x = a.nw = None
    xq = torch.empty(n_tok * (n_in // 256 * 292 if vt == Q8_K else n_in // 32 * 34), dtype=torch.uint8, device=DEV)
    a.xq = xq.data_ptr()
    keep.append(xq)
    if vt == Q8_K and n_tok >= 16 and lib.sdy_gemm_ok(m, n_tok):
        ws = torch.empty(lib.sdy_gemm_ws_bytes(n_tok, n_in), dtype=torch.uint8, device=DEV)
        keep.append(ws)
        a.ws_ready = 1
        if nw is not None:
            xb = torch.empty_like(x)
            keep.append(xb)
            calls.append((lib.sdy_norm_quant_gemm, (xp, nwp, EPS, n_in, n_tok, xb.data_ptr(), a.xq, ws.data_ptr(), None)))
        else:
            calls.append((lib.sdy_quantize_gemm, (xp, a.xq, n_in, n_tok, ws.data_ptr(), None)))
        calls.append((lib.sdy_gemm, (m, arg, ws.data_ptr(), None)))
        return _Calls(calls, out, keep)
    if nw is not None:
        xb = torch.empty_like(x)
        keep.append(xb)
        calls.append((lib.sdy_norm_quant, (xp, nwp, EPS, n_in, n_tok, xb.data_ptr(), vt, a.xq, None)))
    else:
        calls.append((lib.sdy_quantize, (vt, xp, a.xq, n_in, n_tok, None)))
    calls.append((lib.sdy_matvec, (m, arg, None)))
    return _Calls(calls, out, keep)


def _swiglu(y):
    gate, up = y[:, 0::2], y[:, 1::2]
    return gate / (1 + torch.exp(-gate)) * up


def _exact_linear(case, seed):
    raw, x, nw, resid = _linear_inputs(case, seed)
    y = _product(case["wtype"], raw, _norm(x, nw) if nw is not None else x, case["n_in"])
    if case["swiglu"]:
        return _swiglu(y)
    return y + resid.double() if resid is not None else y


def _attention_inputs(case, seed):
    """q, the new token's k and v (decode), and a cache holding `past` positions (a prompt's own ones after them)"""
    g = _gen(seed)
    hd, nkv, n_tok = case["head_dim"], case["n_kv_head"], case.get("n_tok", 1)
    dt = torch.float16 if case["kv"] == "f16" else torch.float32
    kc, vc = (torch.zeros(nkv, case["past"] + n_tok + MAX_SEQ_PAD, hd, device=DEV, dtype=dt) for _ in range(2))
    filled = case["past"] + (n_tok if case["kind"] == "prompt_attention" else 0)
    for c in (kc, vc):
        c[:, :filled] = _randn(g, nkv, filled, hd).to(dt)
    q = _randn(g, n_tok, case["n_head"] * hd)
    k, v = _randn(g, nkv * hd), _randn(g, nkv * hd)
    qn, kn = (torch.empty(hd, device=DEV).uniform_(0.5, 1.5, generator=g) for _ in range(2))
    return q, k, v, kc, vc, qn, kn


def _prepare_prompt_attention(case, seed):
    q, _, _, kc, vc, _, _ = _attention_inputs(case, seed)
    hd, n_tok = case["head_dim"], case["n_tok"]
    out = torch.zeros(n_tok, case["n_head"] * hd, device=DEV)
    kv = capi.KV_F16 if case["kv"] == "f16" else capi.KV_F32
    args = (q.data_ptr(), kc.data_ptr(), vc.data_ptr(), kv, n_tok, case["n_head"], case["n_kv_head"], hd,
            case["past"] + 1, kc.shape[1] * hd, q.shape[1], out.data_ptr(), out.shape[1], None)
    return _Calls([(capi.lib().sdy_attention_flash, args)], out, [q, kc, vc])


def _attend(q, k, v, first):
    """q [T][heads][hd], k and v [kv heads][n][hd] in float64; token t sees positions 0 .. first + t"""
    rep = q.shape[1] // k.shape[0]
    out = torch.empty_like(q)
    see = torch.arange(k.shape[1], device=DEV)[None, :] <= first + torch.arange(q.shape[0], device=DEV)[:, None]
    for h in range(q.shape[1]):
        s = q[:, h] @ k[h // rep].T / math.sqrt(q.shape[2])
        out[:, h] = torch.softmax(s.masked_fill(~see, -math.inf), -1) @ v[h // rep]
    return out


def _exact_prompt_attention(case, seed):
    q, _, _, kc, vc, _, _ = _attention_inputs(case, seed)
    n = case["past"] + case["n_tok"]
    y = _attend(q.double().reshape(case["n_tok"], case["n_head"], -1), kc[:, :n].double(), vc[:, :n].double(),
                case["past"])
    return y.reshape(case["n_tok"], -1)


def _rope_table(n_pos, hd):
    f = 1e6 ** (-torch.arange(0, hd, 2, dtype=torch.float64, device=DEV) / hd)
    a = torch.arange(n_pos, dtype=torch.float64, device=DEV)[:, None] * f
    return torch.cos(a).float(), torch.sin(a).float()


def _rope(x, cos, sin):
    """x [..., hd] in halves"""
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _prepare_decode_attention(case, seed):
    lib = capi.lib()
    q, k, v, kc, vc, qn, kn = _attention_inputs(case, seed)
    hd, nh, nkv, pos, max_seq = case["head_dim"], case["n_head"], case["n_kv_head"], case["past"], kc.shape[1]
    cos, sin = _rope_table(max_seq, hd)
    step = torch.tensor([0, pos], dtype=torch.int32, device=DEV)
    part = torch.empty(lib.sdy_attn_chunked_floats(nh, hd, max_seq), device=DEV)
    out = torch.zeros(nh * hd, device=DEV)
    kv = capi.KV_F16 if case["kv"] == "f16" else capi.KV_F32
    norms = (qn.data_ptr(), kn.data_ptr()) if case["qk_norm"] else (None, None)
    args = (q.data_ptr(), k.data_ptr(), v.data_ptr(), *norms, EPS, cos.data_ptr(), sin.data_ptr(), step.data_ptr(), nh,
            nkv, hd, 0, kc.data_ptr(), vc.data_ptr(), kv, max_seq * hd, max_seq, part.data_ptr(), out.data_ptr(), None,
            None)
    return _Calls([(lib.sdy_attn_decode_chunked, args)], {"out": out, "k": kc[:, pos], "v": vc[:, pos]},
                  [q, k, v, qn, kn, kc, vc, cos, sin, step, part])


def _exact_decode_attention(case, seed):
    q, k, v, kc, vc, qn, kn = _attention_inputs(case, seed)
    hd, pos = case["head_dim"], case["past"]
    q, k, v = (t.double().reshape(-1, hd) for t in (q, k, v))
    if case["qk_norm"]:
        q, k = (t / torch.sqrt((t ** 2).mean(-1, keepdim=True) + EPS) * w.double() for t, w in ((q, qn), (k, kn)))
    cos, sin = (t[pos].double() for t in _rope_table(pos + 1, hd))
    q, k = _rope(q, cos, sin), _rope(k, cos, sin)
    kd, vd = kc[:, :pos + 1].double(), vc[:, :pos + 1].double()
    stored = (k.half().double(), v.half().double()) if case["kv"] == "f16" else (k, v)
    kd[:, pos], vd[:, pos] = stored
    return {"out": _attend(q[None], kd, vd, pos).reshape(-1), "k": stored[0], "v": stored[1]}


# ------------------------------------------------------------------------------------ whole models

def _shape(case):
    if case["arch"] == "qwen3moe":
        return {"dim": 2048, "n_head": 32, "n_kv_head": 4, "hd": 128, "ffn": 768, "experts": 128, "used": 8}
    return {"dim": 2048, "n_head": 16, "n_kv_head": 2, "hd": 128, "ffn": 11008, "experts": 0, "used": 0}


def _model(case, seed):
    """{tensor name: (type, ne, bytes [rows][row bytes])} of the case's model; Q4_K_M files hold attn_v, ffn_down and
    the head in Q6_K"""
    g, s = _gen(seed), _shape(case)
    dim, hd, ffn = s["dim"], s["hd"], s["ffn"]
    q_dim, kv_dim = s["n_head"] * hd, s["n_kv_head"] * hd
    small, large = ("Q4_K", "Q6_K") if case["file"] == "Q4_K_M" else ("Q8_0", "Q8_0")
    t = {}

    def matrix(name, wtype, n_in, rows, experts=0):
        raw = _blocks(wtype, rows * max(1, experts), n_in, g)
        t[name] = (wtype, (n_in, rows, experts) if experts else (n_in, rows), raw)

    def vector(name, n, std=0.0):
        v = _randn(g, n) * std if std else torch.empty(n, device=DEV).uniform_(0.5, 1.5, generator=g)
        t[name] = ("F32", (n,), v.reshape(1, -1).view(torch.uint8))

    matrix("token_embd.weight", small, dim, case["vocab"])
    vector("output_norm.weight", dim)
    matrix("output.weight", large, dim, case["vocab"])
    for l in range(case["n_layer"]):
        p = "blk.%d." % l
        vector(p + "attn_norm.weight", dim)
        vector(p + "ffn_norm.weight", dim)
        matrix(p + "attn_q.weight", small, dim, q_dim)
        matrix(p + "attn_k.weight", small, dim, kv_dim)
        matrix(p + "attn_v.weight", large, dim, kv_dim)
        matrix(p + "attn_output.weight", small, q_dim, dim)
        if s["experts"]:
            vector(p + "attn_q_norm.weight", hd)
            vector(p + "attn_k_norm.weight", hd)
            matrix(p + "ffn_gate_inp.weight", "F32", dim, s["experts"])
            matrix(p + "ffn_gate_exps.weight", small, dim, ffn, s["experts"])
            matrix(p + "ffn_up_exps.weight", small, dim, ffn, s["experts"])
            matrix(p + "ffn_down_exps.weight", large, ffn, dim, s["experts"])
        else:
            for n, d in (("attn_q", q_dim), ("attn_k", kv_dim), ("attn_v", kv_dim)):
                vector(p + n + ".bias", d, 0.1)
            matrix(p + "ffn_gate.weight", small, dim, ffn)
            matrix(p + "ffn_up.weight", small, dim, ffn)
            matrix(p + "ffn_down.weight", large, ffn, dim)
    return t


def _tokens(case, seed):
    r = np.random.default_rng(seed)
    ids = r.integers(0, case["vocab"], case["past"] + case["n_tok"])
    return ids[:case["past"]].astype(np.int32), ids[case["past"]:].astype(np.int32)


def _prepare_engine(case, seed):
    s = _shape(case)
    a = case["arch"]
    with tempfile.TemporaryDirectory(dir="/dev/shm" if os.access("/dev/shm", os.W_OK) else None) as folder:
        b = GGUFBuilder(os.path.join(folder, "model.gguf"))
        b.add_str("general.architecture", a)
        for key, v in (("context_length", 4096), ("embedding_length", s["dim"]), ("block_count", case["n_layer"]),
                       ("feed_forward_length", s["ffn"]), ("attention.head_count", s["n_head"]),
                       ("attention.head_count_kv", s["n_kv_head"]), ("attention.key_length", s["hd"]),
                       ("attention.value_length", s["hd"])):
            b.add_u32("%s.%s" % (a, key), v)
        b.add_f32(a + ".rope.freq_base", 1e6)
        b.add_f32(a + ".attention.layer_norm_rms_epsilon", EPS)
        if s["experts"]:
            b.add_u32(a + ".expert_count", s["experts"])
            b.add_u32(a + ".expert_used_count", s["used"])
            b.add_u32(a + ".expert_feed_forward_length", s["ffn"])
        for name, (wtype, ne, raw) in _model(case, seed).items():
            b.add_tensor(name, ne, wtype, lambda raw=raw: memoryview(raw.cpu().numpy().reshape(-1)))
        model = LoadedModel(b.write())
    past, tokens = _tokens(case, seed)
    session = model.session(max_seq=1536, n_batch=512)
    if past.size:
        session.feed(past)
    return {"session": session, "past": int(past.size), "tokens": tokens, "decode": case["decode"]}


def _run_engine(s):
    s["session"].rewind(s["past"])
    if s["decode"]:
        return [s["session"].step(int(t)) for t in s["tokens"]]
    return s["session"].feed(s["tokens"])


def _exact_engine(case, seed):
    s, t = _shape(case), _model(case, seed)
    past, tokens = _tokens(case, seed)
    ids = torch.from_numpy(np.concatenate([past, tokens]).astype(np.int64)).to(DEV)
    hd, nh, nkv, n = s["hd"], s["n_head"], s["n_kv_head"], ids.numel()
    vec = lambda name: t[name][2].view(torch.float32).reshape(-1)  # noqa: E731

    def mul(name, x, rows=None):
        wtype, ne, raw = t[name]
        return _product(wtype, raw if rows is None else raw[rows[0]:rows[1]], x, ne[0])

    wtype, ne, raw = t["token_embd.weight"]
    x = _values(wtype, raw[ids], ne[0])
    cos, sin = (v.double()[:, None] for v in _rope_table(n, hd))
    for l in range(case["n_layer"]):
        p = "blk.%d." % l
        h = _norm(x, vec(p + "attn_norm.weight"))
        q, k, v = (mul(p + "attn_%s.weight" % c, h) for c in "qkv")
        if not s["experts"]:
            q, k, v = (y + vec(p + "attn_%s.bias" % c).double() for y, c in ((q, "q"), (k, "k"), (v, "v")))
        q, k, v = q.reshape(n, nh, hd), k.reshape(n, nkv, hd), v.reshape(n, nkv, hd)
        if s["experts"]:
            q, k = _norm(q, vec(p + "attn_q_norm.weight")), _norm(k, vec(p + "attn_k_norm.weight"))
        q, k = _rope(q.double(), cos, sin), _rope(k.double(), cos, sin)
        y = _attend(q, k.permute(1, 0, 2).contiguous(), v.permute(1, 0, 2).contiguous(), 0)
        x = x + mul(p + "attn_output.weight", y.reshape(n, -1).float())
        h = _norm(x, vec(p + "ffn_norm.weight"))
        silu_mul = lambda g, u: (g / (1 + torch.exp(-g)) * u).float()  # noqa: E731
        if not s["experts"]:
            x = x + mul(p + "ffn_down.weight", silu_mul(mul(p + "ffn_gate.weight", h), mul(p + "ffn_up.weight", h)))
            continue
        top = torch.softmax(mul(p + "ffn_gate_inp.weight", h), -1).topk(s["used"], -1)
        weight = top.values / top.values.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(s["experts"]):
            at, slot = (top.indices == e).nonzero(as_tuple=True)
            if at.numel():
                rows, down = (e * s["ffn"], (e + 1) * s["ffn"]), (e * s["dim"], (e + 1) * s["dim"])
                u = silu_mul(mul(p + "ffn_gate_exps.weight", h[at], rows), mul(p + "ffn_up_exps.weight", h[at], rows))
                y[at] += weight[at, slot][:, None] * mul(p + "ffn_down_exps.weight", u, down)
        x = x + y
    rows = torch.arange(past.size, n, device=DEV) if case["decode"] else torch.tensor([n - 1], device=DEV)
    y = mul("output.weight", _norm(x[rows], vec("output_norm.weight"))).cpu().numpy()
    return list(y) if case["decode"] else y[0]


# ---------------------------------------------------------------------------------- the interface

def prepare(case, seed):
    capi.check(capi.lib().sdy_init())
    state = {"linear": _prepare_linear, "prompt_attention": _prepare_prompt_attention,
             "decode_attention": _prepare_decode_attention, "engine": _prepare_engine}[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    if isinstance(state, dict):
        return _run_engine(state)
    for call, args in state.calls:
        capi.check(call(*args))
    return state.out


def exact(case, seed):
    return {"linear": _exact_linear, "prompt_attention": _exact_prompt_attention,
            "decode_attention": _exact_decode_attention, "engine": _exact_engine}[case["kind"]](case, seed)


def _weight_bytes(wtype, rows, n_in):
    _, block, size = TYPES[wtype]
    return rows * n_in // block * size


def work(case):
    """Weights, inputs and outputs once each; the multiplications and additions of the products."""
    if case["kind"] == "linear":
        n_in, n_out, n_tok = case["n_in"], case["n_out"], case["n_tok"]
        out = n_tok * (n_out // 2 if case["swiglu"] else n_out)
        floats = n_tok * n_in + out * (2 if case["resid"] else 1) + (n_in if case["norm"] else 0)
        return {"bytes": _weight_bytes(case["wtype"], n_out, n_in) + 4 * floats, "flops": 2 * n_in * n_out * n_tok}
    if case["kind"] != "engine":
        hd, nh, nkv, n_tok = case["head_dim"], case["n_head"], case["n_kv_head"], case.get("n_tok", 1)
        elt = 2 if case["kv"] == "f16" else 4
        pairs = sum(case["past"] + t + 1 for t in range(n_tok))
        return {"bytes": 2 * nkv * (case["past"] + n_tok) * hd * elt + 8 * n_tok * nh * hd,
                "flops": 4 * nh * hd * pairs}
    s, n = _shape(case), case["n_tok"]
    dim, q_dim, kv_dim = s["dim"], s["n_head"] * s["hd"], s["n_kv_head"] * s["hd"]
    small, large = ("Q4_K", "Q6_K") if case["file"] == "Q4_K_M" else ("Q8_0", "Q8_0")
    passes, rows = (n, 1) if case["decode"] else (1, n)  # times the weights are read, tokens each time
    attn = [(small, q_dim + kv_dim, dim), (large, kv_dim, dim), (small, dim, q_dim)]
    if s["experts"]:
        chosen = min(s["experts"], s["used"] * rows)
        experts = [(small, 2 * s["ffn"], dim), (large, dim, s["ffn"])]
        read = attn + [("F32", s["experts"], dim)] + [(w, o * chosen, i) for w, o, i in experts]
        mult = attn + [("F32", s["experts"], dim)] + [(w, o * s["used"], i) for w, o, i in experts]
    else:
        read = mult = attn + [(small, 2 * s["ffn"], dim), (large, dim, s["ffn"])]
    head = [(large, case["vocab"], dim)]
    pairs = sum(case["past"] + t + 1 for t in range(n))
    seen = pairs if case["decode"] else case["past"] + n  # cached positions read
    out = passes * case["vocab"] * 4
    return {"bytes": passes * (case["n_layer"] * sum(_weight_bytes(*w) for w in read) +
                               sum(_weight_bytes(*w) for w in head)) + case["n_layer"] * 8 * kv_dim * seen + out,
            "flops": n * case["n_layer"] * 2 * sum(o * i for _, o, i in mult) +
            passes * 2 * case["vocab"] * dim + case["n_layer"] * 4 * q_dim * pairs}


def tolerance(case):
    if case["kind"] == "linear":
        # 8-bit rows times quantised weights: exact whole-number sums per block, added in 32 bits; float weights: one
        # 32-bit chain of up to 11008 terms, in any order
        return {"rel": 4e-6 if case["wtype"] in FLOAT else 2e-6}
    if case["kind"] != "engine":
        return {"rel": 2e-6 if case["kv"] == "f32" else 4e-6, "max": 1e-3}
    # a last-bit change ahead of a layer moves some activations to the next 8-bit value: against 64-bit attention
    # and norms the decoded logits differ by 1.4e-2
    return {"rel": 3e-2, "max": 0.3}
