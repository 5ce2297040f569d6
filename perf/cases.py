"""What the library's performance is judged on: the work of a program that runs the Qwen3.5 hybrid
decoder on one GPU, call by call, from a single matvec to a whole prompt.

The kernel cases call the C ABI on device pointers (torch tensors) through ``pyq35.lib``, as an
engine that keeps its own buffers does; the model cases go through ``pyq35.Model``. The shapes
are those of the 0.8B- and 2B-shaped models of ``pyq35.dims_for``; weights, caches and states
are random of the distributions those tests and the benchmark use.
"""
from __future__ import annotations

import ctypes as C
import json
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qwen3.5-cpu-cpp_amd"))
import pyq35  # noqa: E402

D = 128          # GDN head dims
HD = 256         # attention head dim
ROT = 64         # rotary dims
THETA = 1e7
EPS = 1e-6
DEV = "cuda"


def listed():
    return [
        # one token's GDN in-projection of the 2B shape: the smallest call of a decode loop
        {"name": "matvec 2B in-projection", "kind": "matvec", "out": 8224, "in": 2048},
        # the delta-rule token of all 18 GDN layers, states resident (an engine that batches layers)
        {"name": "gdn decode 18 layers", "kind": "gdn_decode", "layers": 18, "k_heads": 16, "v_heads": 16, "pos": 1037},
        # one token's attention over an 8k fp32 cache, the 6 layers of the 2B shape
        {"name": "attention decode 2B 8k", "kind": "attn_decode", "layers": 6, "q_heads": 16, "kv_heads": 2,
         "pos": 8191, "max_context": 8256, "bf16": False},
        # the 0.8B shape's GQA group of 4 on a ragged chat-length bf16 cache
        {"name": "attention decode 0.8B 3k bf16", "kind": "attn_decode", "layers": 6, "q_heads": 8, "kv_heads": 2,
         "pos": 3001, "max_context": 4096, "bf16": True},
        # a short chat turn through one projection: fewer tokens than a tile of anything
        {"name": "projection 77 tokens", "kind": "gemm", "M": 77, "N": 8224, "K": 2048, "resid": False},
        # a full block of prompt tokens through the FFN down projection with its residual
        {"name": "projection 4096 tokens", "kind": "gemm", "M": 4096, "N": 2048, "K": 6144, "resid": True},
        # a full block of prompt tokens through one GDN layer
        {"name": "gdn prefill 4096", "kind": "gdn_prefill", "T": 4096, "pos0": 0, "k_heads": 16, "v_heads": 16},
        # a full block of prompt tokens through one attention layer
        {"name": "attention prefill 4096", "kind": "attn_prefill", "T": 4096, "pos0": 0, "q_heads": 16, "kv_heads": 2,
         "max_context": 4096, "bf16": False},
        # a later chat turn: 300 tokens onto 7000 cached positions, 0.8B heads, bf16 cache
        {"name": "attention turn 300 at 7000", "kind": "attn_prefill", "T": 300, "pos0": 7000, "q_heads": 8,
         "kv_heads": 2, "max_context": 8192, "bf16": True},
        # time to the first token of a short prompt on the small model
        {"name": "prompt 32 tokens 0.8B", "kind": "prompt", "model": "0.8b", "tokens": 32, "context": 0, "bf16": False},
        # time to the first token of a long prompt on the 2B shape
        {"name": "prompt 4096 tokens 2B", "kind": "prompt", "model": "2b", "tokens": 4096, "context": 0, "bf16": False},
        # greedy decode at 8k of context on the 2B shape
        {"name": "decode 2B 8k", "kind": "decode", "model": "2b", "context": 8192, "steps": 17, "bf16": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "gdn_decode", "attn_decode", "gemm", "gdn_prefill", "attn_prefill", "prompt", "decode"])
    bf16 = rng.random() < 0.4
    if kind == "matvec":
        return {"kind": kind, "out": _log(rng, 2048, 16384), "in": 8 * _log(rng, 256, 1024)}
    if kind == "gemm":
        return {"kind": kind, "M": _log(rng, 1, 4096), "N": rng.choice([1024, 2048, 5120, 8224, 12288, _log(rng, 256, 8192)]),
                "K": rng.choice([1024, 2048, 3584, 4096, 6144, 8 * _log(rng, 32, 768)]), "resid": rng.random() < 0.5}
    if kind in ("gdn_decode", "gdn_prefill"):
        kh = rng.choice([2, 4, 8, 16, 16])
        vh = kh * (1 if kh == 16 else rng.choice([1, 2]))
        if kind == "gdn_decode":
            return {"kind": kind, "layers": rng.randint(1, 18), "k_heads": kh, "v_heads": vh, "pos": _log(rng, 1, 100000)}
        return {"kind": kind, "T": _log(rng, 1, 4096), "pos0": rng.choice([0, _log(rng, 1, 100000)]), "k_heads": kh,
                "v_heads": vh}
    if kind in ("attn_decode", "attn_prefill"):
        nq, nkv = rng.choice([(16, 2), (16, 2), (8, 2), (8, 2), (4, 1), (2, 1)])
        if kind == "attn_decode":
            pos = _log(rng, 64, 32768)
            return {"kind": kind, "layers": rng.randint(1, 6), "q_heads": nq, "kv_heads": nkv, "pos": pos,
                    "max_context": pos + _log(rng, 1, 4096), "bf16": bf16}
        T, pos0 = _log(rng, 1, 4096), rng.choice([0, _log(rng, 1, 16384)])
        return {"kind": kind, "T": T, "pos0": pos0, "q_heads": nq, "kv_heads": nkv,
                "max_context": pos0 + T + _log(rng, 1, 1024), "bf16": bf16}
    model = rng.choice(["0.8b", "2b"])
    if kind == "prompt":
        ctx = rng.choice([0, 0, _log(rng, 16, 8192)])
        return {"kind": kind, "model": model, "tokens": _log(rng, 2, 2048 if ctx else 4095), "context": ctx, "bf16": bf16}
    return {"kind": kind, "model": model, "context": _log(rng, 16, 32768), "steps": rng.randint(9, 25), "bf16": bf16}


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 12345)
    return g


def _normal(g, *shape, std=1.0, dtype=torch.float32):
    x = torch.empty(shape, dtype=torch.float32, device=DEV)
    x.normal_(0.0, std, generator=g)
    return x if dtype == torch.float32 else x.to(dtype)


def _checkpoint(name):
    """Directory of the named shape's random checkpoint (bf16 N(0, 0.02)), written once per user."""
    path = os.path.join(tempfile.gettempdir(), "q35_cases_%d_%s" % (os.getuid(), name))
    if not os.path.exists(os.path.join(path, "model.safetensors")):
        tmp = tempfile.mkdtemp(prefix="q35_cases_")
        pyq35.synth_write_model(tmp, pyq35.dims_for(name), seed=0, std=0.02)
        try:
            os.rename(tmp, path)
        except OSError:  # written meanwhile by another process
            return path if os.path.exists(os.path.join(path, "model.safetensors")) else tmp
    return path


def _gdn_inputs(g, tokens, kh, vh):
    """Projection rows [q | k | v | z | b | a] of `tokens` tokens, and one layer's small weights."""
    conv = (2 * kh + vh) * D
    return {"proj": _normal(g, tokens, conv + vh * D + 2 * vh), "conv_w": _normal(g, conv, 4, std=0.5),
            "A_log": _normal(g, vh), "dt_bias": _normal(g, vh), "norm_w": 1.0 + _normal(g, D, std=0.1),
            "ring": _normal(g, 4, conv), "state": _normal(g, vh, D, D, std=0.1)}


def _gdn_layers(case, seed):
    g = _gen(seed)
    layers = [_gdn_inputs(g, 1, case["k_heads"], case["v_heads"]) for _ in range(case["layers"])]
    s = {k: torch.stack([x[k] for x in layers]).contiguous() for k in layers[0]}
    kh, vh = case["k_heads"], case["v_heads"]
    conv, p = (2 * kh + vh) * D, s.pop("proj")[:, 0]
    for n, lo, hi in (("qkv", 0, conv), ("z", conv, conv + vh * D), ("b", conv + vh * D, conv + vh * D + vh),
                      ("a", conv + vh * D + vh, conv + vh * D + 2 * vh)):
        s[n] = p[:, lo:hi].contiguous()
    return s


def _attn_inputs(case, seed):
    g = _gen(seed)
    L, NQ, NKV = case.get("layers", 1), case["q_heads"], case["kv_heads"]
    kv = torch.bfloat16 if case["bf16"] else torch.float32
    s = {"k_cache": _normal(g, L, NKV, case["max_context"], HD, dtype=kv),
         "v_cache": _normal(g, L, NKV, case["max_context"], HD, dtype=kv),
         "q_norm": _normal(g, L, HD, std=0.1), "k_norm": _normal(g, L, HD, std=0.1)}
    if case["kind"] == "attn_decode":
        s["qg"], s["k_new"], s["v_new"] = _normal(g, L, NQ, 2 * HD), _normal(g, L, NKV, HD), _normal(g, L, NKV, HD)
    else:
        s["qkv"] = _normal(g, case["T"], 2 * NQ * HD + 2 * NKV * HD)
    return s


def _matrices(case, seed):
    g = _gen(seed)
    if case["kind"] == "matvec":
        return {"W": _normal(g, case["out"], case["in"], std=0.02, dtype=torch.bfloat16), "x": _normal(g, case["in"])}
    s = {"W": _normal(g, case["N"], case["K"], std=0.02, dtype=torch.bfloat16), "X": _normal(g, case["M"], case["K"])}
    if case["resid"]:
        s["R"] = _normal(g, case["M"], case["N"])
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prompt", "decode"):
        return _prepare_model(case, seed)
    new = lambda *n: torch.empty(n, dtype=torch.float32, device=DEV)  # noqa: E731
    if kind in ("matvec", "gemm"):
        s = _matrices(case, seed)
        if kind == "matvec":
            s["y"] = new(case["out"])
        else:
            s["Y"] = new(case["M"], case["N"])
    elif kind == "gdn_decode":
        s = _gdn_layers(case, seed)
        s["out"] = new(case["layers"], case["v_heads"] * D)
        s["args"] = pyq35.GdnDecodeArgs(
            n_layers=case["layers"], k_heads=case["k_heads"], v_heads=case["v_heads"], head_dim_k=D, head_dim_v=D,
            conv_kernel=4, pos=case["pos"], eps=EPS, conv_ring=s["ring"].data_ptr(),
            **{n: s[n].data_ptr() for n in ("qkv", "z", "b", "a", "conv_w", "A_log", "dt_bias", "norm_w", "state", "out")})
    elif kind == "gdn_prefill":
        kh, vh, T = case["k_heads"], case["v_heads"], case["T"]
        s = _gdn_inputs(_gen(seed), T, kh, vh)
        s["out"] = new(T, vh * D)
        ld, conv, base = s["proj"].shape[1], (2 * kh + vh) * D, s["proj"].data_ptr()
        a = pyq35.GdnPrefillArgs(
            n_tokens=T, pos0=case["pos0"], k_heads=kh, v_heads=vh, head_dim_k=D, head_dim_v=D, conv_kernel=4, eps=EPS,
            qkv=base, z=base + 4 * conv, b=base + 4 * (conv + vh * D), a=base + 4 * (conv + vh * D + vh),
            ld_qkv=ld, ld_z=ld, ld_ba=ld, conv_ring=s["ring"].data_ptr(),
            **{n: s[n].data_ptr() for n in ("conv_w", "A_log", "dt_bias", "norm_w", "state", "out")})
        _workspace(s, a, pyq35.lib.q35_gdn_prefill_workspace_bytes)
    else:
        s = _attn_inputs(case, seed)
        T, NQ = case.get("T", 1), case["q_heads"]
        same = dict(q_heads=NQ, kv_heads=case["kv_heads"], head_dim=HD, rotary_dim=ROT, kv_dtype=int(case["bf16"]),
                    max_context=case["max_context"], rope_theta=THETA, eps=EPS,
                    **{n: s[n].data_ptr() for n in ("q_norm", "k_norm", "k_cache", "v_cache")})
        if kind == "attn_decode":
            s["out"] = new(case["layers"], NQ * HD)
            a = pyq35.AttnDecodeArgs(pos=case["pos"], n_splits=0, n_layers=case["layers"], out=s["out"].data_ptr(),
                                     **{n: s[n].data_ptr() for n in ("qg", "k_new", "v_new")}, **same)
            _workspace(s, a, pyq35.lib.q35_attn_decode_workspace_bytes)
        else:
            s["out"] = new(T, NQ * HD)
            a = pyq35.AttnPrefillArgs(n_tokens=T, pos0=case["pos0"], qkv=s["qkv"].data_ptr(), ld_qkv=s["qkv"].shape[1],
                                      out=s["out"].data_ptr(), **same)
            _workspace(s, a, pyq35.lib.q35_attn_prefill_workspace_bytes)
    s["kind"], s["stream"] = kind, torch.cuda.current_stream().cuda_stream
    torch.cuda.current_stream().synchronize()
    return s


def _workspace(s, args, size):
    n = size(C.byref(args))
    s["ws"] = torch.empty(n, dtype=torch.uint8, device=DEV)
    args.workspace, args.workspace_bytes = s["ws"].data_ptr(), n
    s["args"] = args


def _prepare_model(case, seed):
    n, ctx = case.get("tokens", case.get("steps")), case["context"]
    block = case.get("tokens", 0)
    m = pyq35.Model(_checkpoint(case["model"]), ctx + n + 8, kv_bytes_per_elem=2 if case["bf16"] else 4,
                    prefill_block=min(4096, block))
    rng = np.random.RandomState(int(seed) & 0x7FFFFFFF)
    s = {"kind": case["kind"], "m": m, "context": ctx, "steps": case.get("steps", 0),
         "ids": rng.randint(0, m.dims.vocab_size, n).astype(np.int32)}
    if ctx:
        m.fill_synthetic(ctx, seed=int(seed), state_std=0.1)
    return s


# --------------------------------------------------------------------------------- run
def run(s):
    kind, lib = s["kind"], pyq35.lib
    if kind == "matvec":
        W = s["W"]
        pyq35.check(lib.q35_matmul_bf16(W.data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(), W.shape[0], W.shape[1],
                                        s["stream"]))
        return s["y"]
    if kind == "gemm":
        X, W, Y, R = s["X"], s["W"], s["Y"], s.get("R")
        M, K, N = X.shape[0], X.shape[1], W.shape[0]
        pyq35.check(lib.q35_gemm_bf16(X.data_ptr(), K, W.data_ptr(), M, N, K, R.data_ptr() if R is not None else None,
                                      N if R is not None else 0, Y.data_ptr(), N, s["stream"]))
        return Y
    if kind == "gdn_decode":
        pyq35.check(lib.q35_gdn_decode(C.byref(s["args"]), s["stream"]))
        return {"out": s["out"], "state": s["state"], "ring": s["ring"]}
    if kind == "gdn_prefill":
        pyq35.check(lib.q35_gdn_prefill(C.byref(s["args"]), s["stream"]))
        return {"out": s["out"], "state": s["state"], "ring": s["ring"]}
    if kind in ("attn_decode", "attn_prefill"):
        fn = lib.q35_attn_decode if kind == "attn_decode" else lib.q35_attn_prefill
        pyq35.check(fn(C.byref(s["args"]), s["stream"]))
        return {"out": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    m, ids = s["m"], s["ids"]
    if kind == "prompt":
        if s["context"]:  # a later turn; the answer before it is dropped
            m.set_position(s["context"])
            m.extend(ids[:-1], want_logits=False)
        else:
            m.prefill(ids[:-1], want_logits=False)
        return m.step(int(ids[-1]))[0]
    m.set_position(s["context"])  # the answer is generated anew
    out = m.decode_greedy(int(ids[0]), s["steps"] - 1)
    return {"ids": out, "logits": m.step(int(out[-1]))[0]}


# --------------------------------------------------------------------- bytes and operations
def _gdn_work(tokens, kh, vh, calls=1):
    """Per layer: rows in and out, the state read and written, and the four matrix-vector passes
    of the recurrence (decay, S^T k, rank-1 update, S^T q: 7 operations a state element)."""
    conv = (2 * kh + vh) * D
    b = 4 * (tokens * (conv + 2 * vh * D + 2 * vh) + calls * (2 * vh * D * D + 4 * conv + 2 * 3 * conv))
    return b, 7.0 * tokens * vh * D * D


def _attn_work(tokens, pos0, nq, nkv, elem):
    keys = tokens * pos0 + tokens * (tokens + 1) / 2
    b = 2 * nkv * HD * elem * (pos0 + tokens) + 4 * tokens * (3 * nq + 2 * nkv) * HD + 2 * nkv * HD * elem * tokens
    return b, 4.0 * nq * HD * keys


def _model_work(case, tokens, pos0):
    """One pass of `tokens` tokens: every projection weight once, the mixers, no output head."""
    d = pyq35.dims_for(case["model"])
    H, I, kh, vh, nq, nkv = (d.hidden_size, d.ffn_intermediate, d.gdn_k_heads, d.gdn_v_heads, d.attn_q_heads,
                             d.attn_kv_heads)
    elem = 2 if case["bf16"] else 4
    pg = H * ((2 * kh + vh) * D + 2 * vh * D + 2 * vh)
    pa = H * (3 * nq + 2 * nkv) * HD
    params = d.n_layers_gdn * pg + d.n_layers_attn * pa + d.n_layers_total * 3 * H * I
    bg, fg = _gdn_work(tokens, kh, vh)
    ba, fa = _attn_work(tokens, pos0, nq, nkv, elem)
    keep = 4 * 2 * d.gdn_v_heads * D * D  # of a block's rows only the state and the cache reach memory
    kv = 2 * nkv * HD * elem * (pos0 + 2 * tokens)
    return (2.0 * params + d.n_layers_gdn * min(bg, keep) + d.n_layers_attn * min(ba, kv),
            2.0 * params * tokens + d.n_layers_gdn * fg + d.n_layers_attn * fa)


def _head_work(case):
    d = pyq35.dims_for(case["model"])
    n = d.hidden_size * d.vocab_size
    return 2.0 * n + 4 * d.vocab_size, 2.0 * n


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        n = case["out"] * case["in"]
        b, f = 2 * n + 4 * (case["out"] + case["in"]), 2.0 * n
    elif kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        b, f = 2 * N * K + 4 * M * K + 4 * M * N * (2 if case["resid"] else 1), 2.0 * M * N * K
    elif kind == "gdn_decode":
        b, f = _gdn_work(1, case["k_heads"], case["v_heads"])
        b, f = b * case["layers"], f * case["layers"]
    elif kind == "gdn_prefill":
        b, f = _gdn_work(case["T"], case["k_heads"], case["v_heads"])
    elif kind in ("attn_decode", "attn_prefill"):
        b, f = _attn_work(case.get("T", 1), case.get("pos0", case.get("pos")), case["q_heads"], case["kv_heads"],
                          2 if case["bf16"] else 4)
        b, f = b * case.get("layers", 1), f * case.get("layers", 1)
    elif kind == "prompt":
        b, f = _model_work(case, case["tokens"], case["context"])
        hb, hf = _head_work(case)
        b, f = b + hb, f + hf
    else:
        b = f = 0.0
        hb, hf = _head_work(case)
        for i in range(case["steps"]):  # each step waits for the last one's token
            sb, sf = _model_work(case, 1, case["context"] + i)
            b, f = b + sb + hb, f + sf + hf
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("matvec", "gemm"):
        # fp32 sums of up to 8192 products in another order
        return {"rel": 2e-6, "max": 5e-5}
    if kind == "gdn_decode":
        return {"rel": 5e-6, "max": 2e-4}
    if kind == "gdn_prefill":
        # the recurrence in chunks of another size, or token by token
        return {"rel": 1e-5, "max": 1e-3}
    if kind in ("attn_decode", "attn_prefill"):
        # bf16: an appended element at a rounding midpoint may round the other way (2^-8 of itself)
        return {"rel": 2e-4, "max": 1e-2} if case["bf16"] else {"rel": 5e-6, "max": 2e-4}
    # 24 layers on
    return {"rel": 4e-4, "max": 4e-3, "differ": 0.0} if case["bf16"] else {"rel": 2e-5, "max": 4e-4, "differ": 0.0}


# ---------------------------------------------------------------------- the same in 64 bits
def _f(x):
    return x.to(torch.float64)


def _gdn64(p, conv_w, A_log, dt_bias, norm_w, window, S, eps, kh, vh):
    """One GDN layer over the projection rows p [T][q|k|v|z|b|a]; window [3][CONV] oldest first."""
    T, kd, vd = p.shape[0], kh * D, vh * D
    conv = 2 * kd + vd
    x = torch.cat([window, p[:, :conv]])
    y = torch.nn.functional.silu(sum(x[i:i + T] * conv_w[:, i] for i in range(4)))
    rep = vh // kh
    unit = lambda v: v / torch.sqrt((v * v).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q = (unit(y[:, :kd].view(T, kh, D)) * D ** -0.5).repeat_interleave(rep, 1)
    k = unit(y[:, kd:2 * kd].view(T, kh, D)).repeat_interleave(rep, 1)
    v = y[:, 2 * kd:].view(T, vh, D)
    z, b, a = p[:, conv:conv + vd].view(T, vh, D), p[:, conv + vd:conv + vd + vh], p[:, conv + vd + vh:conv + vd + 2 * vh]
    alpha = torch.exp(-torch.exp(A_log) * torch.nn.functional.softplus(a + dt_bias))[:, :, None, None]
    beta = torch.sigmoid(b)[:, :, None, None]
    S = S.clone()
    o = torch.empty_like(v)
    kc, kr, vr, qr = k[:, :, :, None], k[:, :, None, :], v[:, :, None, :], q[:, :, None, :]
    for t in range(T):
        S *= alpha[t]
        S.baddbmm_(kc[t], (vr[t] - torch.bmm(kr[t], S)) * beta[t])
        o[t] = torch.bmm(qr[t], S)[:, 0]
    n = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + eps) * norm_w * torch.nn.functional.silu(z)
    return n.reshape(T, vd), S, x[T:]


def _rope64(x, pos):
    inv = THETA ** (-torch.arange(0, ROT, 2, dtype=torch.float64, device=x.device) / ROT)
    ang = pos.to(torch.float64)[:, None, None] * inv
    c, s, h = torch.cos(ang), torch.sin(ang), ROT // 2
    a, b = x[..., :h], x[..., h:ROT]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., ROT:]], -1)


def _attn64(qg, k, v, q_norm, k_norm, kc, vc, pos0, eps, bf16):
    """qg [T][NQ][2 HD], k / v [T][NKV][HD]; appends to the float64 caches [NKV][ctx][HD] in place."""
    T, nq, nkv = qg.shape[0], qg.shape[1], k.shape[1]
    pos = torch.arange(pos0, pos0 + T, device=qg.device)
    norm = lambda x, w: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 + w)  # noqa: E731
    cut = (lambda x: _f(x.to(torch.bfloat16))) if bf16 else (lambda x: x)
    q = _rope64(norm(qg[..., :HD], q_norm), pos)
    kc[:, pos0:pos0 + T] = cut(_rope64(norm(k, k_norm), pos)).transpose(0, 1)
    vc[:, pos0:pos0 + T] = cut(v).transpose(0, 1)
    out = torch.empty(T, nq, HD, dtype=torch.float64, device=qg.device)
    hide = torch.arange(pos0 + T, device=qg.device)[None, :] > pos[:, None]
    for h in range(nq):
        K, V = kc[h * nkv // nq, :pos0 + T], vc[h * nkv // nq, :pos0 + T]
        w = torch.softmax((q[:, h] @ K.T.contiguous() * HD ** -0.5).masked_fill_(hide, -math.inf), -1)
        out[:, h] = w @ V * torch.sigmoid(qg[:, h, HD:])
    return out.reshape(T, nq * HD)


def _window(ring, pos):
    return torch.stack([ring[(pos - 3 + i) % 4] for i in range(3)])


def exact(case, seed):
    kind = case["kind"]
    if kind == "matvec":
        s = _matrices(case, seed)
        return _f(s["W"]) @ _f(s["x"])
    if kind == "gemm":
        s = _matrices(case, seed)
        y = _f(s["X"]) @ _f(s["W"]).T.contiguous()
        return y + _f(s["R"]) if case["resid"] else y
    if kind == "gdn_decode":
        s = _gdn_layers(case, seed)
        kh, vh, pos, out, st = case["k_heads"], case["v_heads"], case["pos"], [], []
        ring = _f(s["ring"])
        for i in range(case["layers"]):
            p = _f(torch.cat([s[n][i] for n in ("qkv", "z", "b", "a")]))[None]
            o, S, _ = _gdn64(p, *(_f(s[n][i]) for n in ("conv_w", "A_log", "dt_bias", "norm_w")),
                             _window(ring[i], pos), _f(s["state"][i]), EPS, kh, vh)
            ring[i, pos % 4] = p[0, :ring.shape[2]]
            out.append(o[0])
            st.append(S)
        return {"out": torch.stack(out), "state": torch.stack(st), "ring": ring}
    if kind == "gdn_prefill":
        kh, vh = case["k_heads"], case["v_heads"]
        s = {k: _f(x) for k, x in _gdn_inputs(_gen(seed), case["T"], kh, vh).items()}
        o, S, _ = _gdn64(s["proj"], s["conv_w"], s["A_log"], s["dt_bias"], s["norm_w"], _window(s["ring"], case["pos0"]),
                         s["state"], EPS, kh, vh)
        ring = s["ring"]  # the slots (position % 4) of the last three rows
        for t in range(max(0, case["T"] - 3), case["T"]):
            ring[(case["pos0"] + t) % 4] = s["proj"][t, :ring.shape[1]]
        return {"out": o, "state": S, "ring": ring}
    if kind in ("attn_decode", "attn_prefill"):
        s = {k: _f(x) for k, x in _attn_inputs(case, seed).items()}
        nq, nkv, outs = case["q_heads"], case["kv_heads"], []
        for i in range(case.get("layers", 1)):
            if kind == "attn_decode":
                rows = s["qg"][i][None], s["k_new"][i][None], s["v_new"][i][None]
            else:
                x, T = s["qkv"], case["T"]
                rows = (x[:, :2 * nq * HD].view(T, nq, 2 * HD), x[:, 2 * nq * HD:(2 * nq + nkv) * HD].view(T, nkv, HD),
                        x[:, (2 * nq + nkv) * HD:].view(T, nkv, HD))
            outs.append(_attn64(*rows, s["q_norm"][i], s["k_norm"][i], s["k_cache"][i], s["v_cache"][i],
                                case.get("pos0", case.get("pos")), EPS, case["bf16"]))
        out = torch.cat(outs) if kind == "attn_decode" else outs[0]
        return {"out": out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "prompt" and not case["context"]:
        return _prompt64(case, seed)
    return None  # a cache and state of the library's own making


class _Weights:
    """The checkpoint's tensors by name, in 64 bits on the GPU (a safetensors file holds a JSON
    table of byte ranges behind its 8-byte length, then the bytes)."""

    def __init__(self, path):
        with open(path, "rb") as f:
            n = struct.unpack("<Q", f.read(8))[0]
            self.table = json.loads(f.read(n))
        self.data = np.memmap(path, np.uint8, "r", offset=8 + n)

    def __call__(self, name):
        t = self.table["model.language_model." + name]
        raw = np.array(self.data[t["data_offsets"][0]:t["data_offsets"][1]])
        return _f(torch.from_numpy(raw.view(np.int16)).to(DEV).view(torch.bfloat16).view(t["shape"]))


def _prompt64(case, seed):
    d = pyq35.dims_for(case["model"])
    w = _Weights(os.path.join(_checkpoint(case["model"]), "model.safetensors"))
    rng = np.random.RandomState(int(seed) & 0x7FFFFFFF)
    ids = torch.from_numpy(rng.randint(0, d.vocab_size, case["tokens"])).to(DEV)
    kh, vh, nq, nkv, T, eps = d.gdn_k_heads, d.gdn_v_heads, d.attn_q_heads, d.attn_kv_heads, len(ids), d.rms_norm_eps
    norm = lambda x, g: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 + g)  # noqa: E731
    lin = lambda x, name: x @ w(name).T.contiguous()  # noqa: E731
    emb = w("embed_tokens.weight")
    x = emb[ids]
    for i in range(d.n_layers_total):
        p = "layers.%d." % i
        y = norm(x, w(p + "input_layernorm.weight"))
        if (i + 1) % d.attn_interval:
            a = p + "linear_attn."
            rows = torch.cat([lin(y, a + n + ".weight") for n in ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a")], 1)
            conv = (2 * kh + vh) * D
            o, _, _ = _gdn64(rows, w(a + "conv1d.weight").view(conv, 4), w(a + "A_log"), w(a + "dt_bias"),
                             w(a + "norm.weight"), rows.new_zeros(3, conv), rows.new_zeros(vh, D, D), eps, kh, vh)
            x = x + lin(o, a + "out_proj.weight")
        else:
            a = p + "self_attn."
            kc, vc = x.new_zeros(nkv, T, HD), x.new_zeros(nkv, T, HD)
            o = _attn64(lin(y, a + "q_proj.weight").view(T, nq, 2 * HD), lin(y, a + "k_proj.weight").view(T, nkv, HD),
                        lin(y, a + "v_proj.weight").view(T, nkv, HD), w(a + "q_norm.weight"), w(a + "k_norm.weight"),
                        kc, vc, 0, eps, case["bf16"])
            x = x + lin(o, a + "o_proj.weight")
        y = norm(x, w(p + "post_attention_layernorm.weight"))
        x = x + lin(torch.nn.functional.silu(lin(y, p + "mlp.gate_proj.weight")) * lin(y, p + "mlp.up_proj.weight"),
                    p + "mlp.down_proj.weight")
    return (norm(x[-1], w("norm.weight")) @ emb.T.contiguous()).cpu().numpy()
