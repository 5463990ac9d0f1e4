"""The work that programs have this library do, as timed cases.

A case is one call pattern through the C ABI (include/kq_gemv.h) on synthetic
weights with the magnitudes of a trained model (|w| around 0.02, scales and
mins that centre the weights) and hidden states as they leave an RMSNorm
(N(0, 1) with a few channels several times larger).  Kinds:

  host   the reference's own signature: host x in, host y out, synchronous
  layer  one decoder layer's matvecs of a decode step, the launches a
         device-resident decode loop issues: [Q, K, V], [O + residual],
         [gate, up], [down + residual]
  gemv   single tensors, one call each (LM head, layers stored in other types)
  multi  B token streams through one weight pass: prefill chunks, speculative
         and batched decode; exact, in the int8-activation mode, or on the
         fp16 matrix cores
  moe    the expert FFN step of MoE layers: router, top-k, expert matvecs,
         SwiGLU, weighted sum

Every pass reads enough distinct weights that, over the states a timing loop
rotates, they do not stay in the 256 MB cache in front of HBM: a decode step
never finds a layer's weights there.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import stratum_amd as KQ

DEV = "cuda"
TYPES = {"Q4_K": KQ.TYPE_Q4_K, "Q6_K": KQ.TYPE_Q6_K, "Q5_K": KQ.TYPE_Q5_K, "Q3_K": KQ.TYPE_Q3_K,
         "Q8_0": KQ.TYPE_Q8_0, "Q2_K": KQ.TYPE_Q2_K, "NIB": KQ.TYPE_Q2K_NIB}
INT8 = ("Q4_K", "Q6_K", "Q5_K", "Q3_K", "Q8_0")


# ------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest call: one matvec through the reference's host signature
        {"name": "host_q4k_1024x1024", "kind": "host", "type": "Q4_K", "N": 1024, "K": 1024, "int8": False},
        # a small model's decode step (0.6B class: hidden 1024, FFN 3072), where
        # launches and latency count; twelve layers so that weights come from HBM
        {"name": "layer_0.6b", "kind": "layer", "H": 1024, "Q": 2048, "KV": 1024, "F": 3072, "L": 12,
         "type": "Q4_K", "down": "Q6_K", "int8": False},
        # the headline: one layer of a 27B-class dense model, one token
        {"name": "layer_27b", "kind": "layer", "H": 5120, "Q": 6144, "KV": 1024, "F": 17408, "L": 1,
         "type": "Q4_K", "down": "Q6_K", "int8": False},
        # the same in the int8-activation mode, the reference's default arithmetic
        {"name": "layer_27b_int8", "kind": "layer", "H": 5120, "Q": 6144, "KV": 1024, "F": 17408, "L": 1,
         "type": "Q4_K", "down": "Q6_K", "int8": True},
        # the LM head of a decode step: many short rows
        {"name": "head_q6k_151936x1024", "kind": "gemv", "type": "Q6_K", "N": 151936, "K": 1024, "n": 1,
         "int8": False},
        # layers kept in a wider type, with a row count that divides nothing
        {"name": "gemv_q5k_11007x4096", "kind": "gemv", "type": "Q5_K", "N": 11007, "K": 4096, "n": 8,
         "int8": False},
        # eight streams through a layer's gate and up (batched decode, exact)
        {"name": "multi_q4k_b8", "kind": "multi", "type": "Q4_K", "N": 17408, "K": 5120, "n": 2, "B": 8,
         "mode": "exact"},
        # an odd number of streams through the long-row down projection, exact
        {"name": "multi_q6k_b13", "kind": "multi", "type": "Q6_K", "N": 5120, "K": 17408, "n": 2, "B": 13,
         "mode": "exact"},
        # sixteen streams in the int8 mode
        {"name": "multi_int8_q4k_b16", "kind": "multi", "type": "Q4_K", "N": 17408, "K": 5120, "n": 2, "B": 16,
         "mode": "int8"},
        # the largest batch of one call on the fp16 matrix cores (a prefill chunk)
        {"name": "multi_mfma_q4k_b64", "kind": "multi", "type": "Q4_K", "N": 17408, "K": 5120, "n": 2, "B": 64,
         "mode": "mfma"},
        # MoE decode, one token: 128 experts, top-8, eight layers
        {"name": "moe_b1", "kind": "moe", "H": 2048, "F": 768, "E": 128, "k": 8, "B": 1, "L": 8,
         "type": "Q4_K", "down": "Q4_K", "int8": False},
        # MoE batched decode, sixteen tokens
        {"name": "moe_b16", "kind": "moe", "H": 2048, "F": 768, "E": 128, "k": 8, "B": 16, "L": 2,
         "type": "Q4_K", "down": "Q4_K", "int8": False},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _k(rng, lo, hi):
    """A row length: a multiple of the 256-weight super-block."""
    return 256 * max(1, round(_log(rng, lo, hi) / 256))


# no drawn case is larger than the largest listed one of its kind of arithmetic
MOST_BYTES, MOST_FLOPS = 4.4e8, {"exact": 4.7e9, "int8": 1.1e10, "mfma": 2.3e10}


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS[c.get("mode", "exact")]:
            return c


def _draw(rng):
    kind = rng.choice(["host", "layer", "gemv", "gemv", "multi", "multi", "multi", "moe", "moe"])
    if kind == "host":
        t = rng.choice(list(TYPES))
        return {"kind": kind, "type": t, "N": int(_log(rng, 32, 18000)), "K": _k(rng, 256, 6144),
                "int8": t in INT8 and rng.random() < 0.4}
    if kind == "layer":
        H = _k(rng, 1024, 5120)
        return {"kind": kind, "H": H, "Q": 256 * max(1, round(H * rng.uniform(1, 2) / 256)),
                "KV": 128 * rng.randint(1, 8), "F": 256 * round(H * rng.uniform(2.5, 3.5) / 256),
                "L": max(1, min(12, int(5120 * 5120 * 1.2 / (H * H)))), "type": rng.choice(["Q4_K", "Q4_K", "Q5_K"]),
                "down": rng.choice(["Q6_K", "Q4_K", "Q8_0"]), "int8": rng.random() < 0.4}
    if kind == "gemv":
        t = rng.choice(list(TYPES))
        K, N = _k(rng, 512, 17408), int(_log(rng, 700, 32000))
        n = max(1, min(8, int(1.2e8 / (N * K))))
        return {"kind": kind, "type": t, "N": N, "K": K, "n": n, "int8": t in INT8 and rng.random() < 0.4}
    if kind == "multi":
        mode = rng.choice(["exact", "exact", "int8", "mfma"])
        t = rng.choice(["Q4_K", "Q4_K", "Q6_K"] if mode == "mfma" else list(INT8) + ["Q4_K", "Q6_K"])
        return {"kind": kind, "type": t, "N": int(_log(rng, 1000, 17408)), "K": _k(rng, 1024, 17408), "n": 2,
                "B": int(_log(rng, 16, 65)) if mode == "mfma" else int(_log(rng, 2, 33)), "mode": mode}
    E = rng.choice([32, 60, 64, 128])
    return {"kind": kind, "H": _k(rng, 1024, 4096), "F": 256 * rng.randint(2, 6), "E": E,
            "k": rng.choice([2, 4, 6, 8]), "B": int(_log(rng, 1, 33)), "L": 2, "type": rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q5_K"]),
            "down": rng.choice(["Q4_K", "Q6_K"]), "int8": rng.random() < 0.5}


# ------------------------------------------- synthetic weights (on the GPU)

def _rand(g, n, hi):
    return torch.randint(0, hi, (n,), generator=g, device=DEV, dtype=torch.uint8)


def _bytes(t):
    """fp16 tensor -> its two little-endian bytes per value."""
    return t.contiguous().view(torch.uint8).reshape(t.shape[0], -1)


def _dscale(g, n, v):
    """Block scales around v: log-normal, as fp16."""
    z = torch.randn(n, generator=g, device=DEV)
    return (v * torch.exp(0.3 * z)).to(torch.float16).reshape(n, 1)


def _pack_scales(sc, m):
    """The 12 scale bytes of Q4_K / Q5_K: 6-bit scales and mins, [n, 8] each."""
    out = torch.empty(sc.shape[0], 12, dtype=torch.uint8, device=DEV)
    out[:, 0:4] = sc[:, 0:4] | ((sc[:, 4:8] >> 4) << 6)
    out[:, 4:8] = m[:, 0:4] | ((m[:, 4:8] >> 4) << 6)
    out[:, 8:12] = (sc[:, 4:8] & 15) | ((m[:, 4:8] & 15) << 4)
    return out


def _blocks(g, t, n):
    """n super-blocks of 256 weights of type t, std about 0.02, mean about 0."""
    if t in ("Q4_K", "Q5_K"):
        half = 7.5 if t == "Q4_K" else 15.5
        sc = 24 + _rand(g, n * 8, 40).reshape(n, 8)
        m = torch.clamp(sc.to(torch.int16) + _rand(g, n * 8, 9).reshape(n, 8).to(torch.int16) - 4, 0, 63).to(torch.uint8)
        d = _dscale(g, n, 0.02 / (43 * half * 0.61))
        body = 128 if t == "Q4_K" else 160
        return torch.cat([_bytes(d), _bytes((d.float() * half).to(torch.float16)), _pack_scales(sc, m),
                          _rand(g, n * body, 256).reshape(n, body)], 1)
    if t == "Q6_K":
        s = (40 + _rand(g, n * 16, 88)).reshape(n, 16).to(torch.int16)
        s = torch.where(_rand(g, n * 16, 2).reshape(n, 16) > 0, s, -s).to(torch.int8).view(torch.uint8)
        return torch.cat([_rand(g, n * 192, 256).reshape(n, 192), s, _bytes(_dscale(g, n, 0.02 / (18.5 * 84)))], 1)
    if t == "Q3_K":
        return torch.cat([_rand(g, n * 108, 256).reshape(n, 108), _bytes(_dscale(g, n, 0.02 / (18.5 * 2.3)))], 1)
    if t == "Q8_0":
        b = torch.cat([_bytes(_dscale(g, 8 * n, 0.02 / 74)), _rand(g, n * 256, 256).reshape(8 * n, 32)], 1)
        return b.reshape(n, 272)
    sc = 4 + _rand(g, n * 16, 12).reshape(n, 16)
    scm = sc | (torch.clamp(sc, 0, 15) << 4)
    d = _dscale(g, n, 0.02 / (9.5 * 1.1))
    dd = torch.cat([_bytes(d), _bytes((d.float() * 1.5).to(torch.float16))], 1)
    if t == "Q2_K":
        return torch.cat([scm, _rand(g, n * 64, 256).reshape(n, 64), dd], 1)
    q = _rand(g, n * 256, 4).reshape(n, 2, 128)       # NIB: two 2-bit values, one per nibble
    return torch.cat([scm, q[:, 0] | (q[:, 1] << 4), dd], 1)


def _weights(seed, salt, t, rows, K):
    """rows x K weights as one uint8 tensor of rows*(K/256) blocks."""
    g = torch.Generator(device=DEV).manual_seed(seed * 1000003 + salt)
    return _blocks(g, t, rows * (K // 256)).contiguous().reshape(-1)


def _x(seed, salt, *shape):
    """Normed hidden states: N(0, 1), one channel in about 200 several times larger."""
    g = torch.Generator(device=DEV).manual_seed(seed * 1000003 + 500009 + salt)
    x = torch.randn(*shape, generator=g, device=DEV)
    big = torch.rand(shape[-1], generator=g, device=DEV) < 0.005
    return torch.where(big, x * 8, x).contiguous()


def _row(t, K):
    return K // 256 * KQ.BLOCK_BYTES[TYPES[t]]


def _id(t, int8):
    return TYPES[t] | (KQ.INT8_ACT if int8 and t in INT8 else 0)


# ------------------------------------------------------------- state and run

_HOST = {}   # (type, N, K) -> registered host weights: uploaded once, as a program does at start-up


def _host_weights(t, N, K):
    """The process's one weight file: kq_linear_init may replace it, so every
    (type, N, K) asked for so far lies in one registered mapping."""
    key = (t, N, K)
    if key not in _HOST:
        _HOST[key] = _weights(7, 0, t, N, K).cpu().numpy()
        offs, blob, at = {}, [], 0
        for k, w in _HOST.items():
            offs[k] = at
            pad = -len(w) % 256
            blob += [w, np.zeros(pad, np.uint8)]
            at += len(w) + pad
        _host_weights.region = KQ.WeightRegion(np.concatenate(blob))
        _host_weights.offs = offs
    return _host_weights.offs[key]


def _segs(*segs):
    return (KQ.KqSegment * len(segs))(*segs)


def prepare(case, seed):
    c, L = dict(case), KQ.lib()
    kind = c["kind"]
    st = {"case": c, "lib": L, "stream": torch.cuda.current_stream().cuda_stream}
    if kind == "host":
        off = _host_weights(c["type"], c["N"], c["K"])
        st["tensor"] = KQ.make_tensor(TYPES[c["type"]], c["N"], c["K"], off)
        st["x"] = _x(seed, 1, c["K"]).cpu().numpy()
        st["y"] = np.empty(c["N"], np.float32)
        F = ctypes.POINTER(ctypes.c_float)
        st["args"] = (ctypes.byref(st["tensor"]), st["x"].ctypes.data_as(F), st["y"].ctypes.data_as(F), c["N"], c["K"])
    elif kind == "layer":
        H, Q, KV, F, n = c["H"], c["Q"], c["KV"], c["F"], c["L"]
        t, td = c["type"], c["down"]
        it, idn = _id(t, c["int8"]), _id(td, c["int8"])
        w = {"qkv": _weights(seed, 1, t, n * (Q + 2 * KV), H), "o": _weights(seed, 2, t, n * H, Q),
             "gu": _weights(seed, 3, t, n * 2 * F, H), "d": _weights(seed, 4, td, n * H, F)}
        x = {"h": _x(seed, 5, n, H), "a": _x(seed, 6, n, Q), "h2": _x(seed, 7, n, H), "f": _x(seed, 8, n, F),
             "r": _x(seed, 9, n, H)}
        y = {"qkv": torch.empty(n, Q + 2 * KV, device=DEV), "o": torch.empty(n, H, device=DEV),
             "gu": torch.empty(n, 2 * F, device=DEV), "d": torch.empty(n, H, device=DEV)}
        rb, calls = _row(t, H), []

        def at(buf, i):
            return buf.data_ptr() + 4 * i * buf.shape[1]

        for i in range(n):
            wq, yq, xh = w["qkv"].data_ptr() + i * (Q + 2 * KV) * rb, at(y["qkv"], i), at(x["h"], i)
            calls.append(_segs(KQ.segment(it, H, Q, [wq], xh, yq), KQ.segment(it, H, KV, [wq + Q * rb], xh, yq + 4 * Q),
                               KQ.segment(it, H, KV, [wq + (Q + KV) * rb], xh, yq + 4 * (Q + KV))))
            calls.append(_segs(KQ.segment(it, Q, H, [w["o"].data_ptr() + i * H * _row(t, Q)], at(x["a"], i),
                                          at(y["o"], i), add_ptr=at(x["r"], i))))
            wg, yg, x2 = w["gu"].data_ptr() + i * 2 * F * rb, at(y["gu"], i), at(x["h2"], i)
            calls.append(_segs(KQ.segment(it, H, F, [wg], x2, yg), KQ.segment(it, H, F, [wg + F * rb], x2, yg + 4 * F)))
            calls.append(_segs(KQ.segment(idn, F, H, [w["d"].data_ptr() + i * H * _row(td, F)], at(x["f"], i),
                                          at(y["d"], i), add_ptr=at(x["r"], i))))
        st.update(w=w, x=x, y=y, calls=[(a, len(a)) for a in calls])
    elif kind == "gemv":
        n, N, K = c["n"], c["N"], c["K"]
        st["w"] = _weights(seed, 1, c["type"], n * N, K)
        st["x"], st["y"] = _x(seed, 2, n, K), torch.empty(n, N, device=DEV)
        rb = N * _row(c["type"], K)
        st["calls"] = [(_id(c["type"], c["int8"]), st["w"].data_ptr() + i * rb, st["x"].data_ptr() + 4 * i * K, None,
                        st["y"].data_ptr() + 4 * i * N, N, K, st["stream"]) for i in range(n)]
    elif kind == "multi":
        n, N, K, B = c["n"], c["N"], c["K"], c["B"]
        st["w"] = _weights(seed, 1, c["type"], n * N, K)
        st["x"], st["y"] = _x(seed, 2, B, K), torch.empty(n, B, N, device=DEV)
        st["fn"] = L.kq_gemv_multix_mfma_dev if c["mode"] == "mfma" else L.kq_gemv_multix_dev
        t, rb = _id(c["type"], c["mode"] == "int8"), N * _row(c["type"], K)
        st["calls"] = [(t, st["w"].data_ptr() + i * rb, st["x"].data_ptr(), st["y"].data_ptr() + 4 * i * B * N, B, N, K,
                        st["stream"]) for i in range(n)]
    else:
        H, F, E, B, n, k = c["H"], c["F"], c["E"], c["B"], c["L"], c["k"]
        t, td = c["type"], c["down"]
        st["w"] = {"g": _weights(seed, 1, t, n * E * F, H), "u": _weights(seed, 2, t, n * E * F, H),
                   "d": _weights(seed, 3, td, n * E * H, F)}
        st["router"] = _x(seed, 4, n, E, H) * 0.03
        st["xn"], st["res"] = _x(seed, 5, n, B, H), _x(seed, 6, n, B, H)
        st["x"] = torch.empty(n, B, H, device=DEV)
        st["sel"] = torch.empty(n, B, k, dtype=torch.int32, device=DEV)
        st["selw"] = torch.empty(n, B, k, device=DEV)
        sg, sd, fs = F * _row(t, H), H * _row(td, F), []
        for i in range(n):
            f = KQ.KqMoeFfn()
            f.n_embed, f.n_ff, f.n_experts, f.k = H, F, E, k
            f.router_type, f.router = KQ.TYPE_F32, st["router"].data_ptr() + 4 * i * E * H
            f.gate_type = f.up_type = _id(t, c["int8"])
            f.down_type = _id(td, c["int8"])
            f.gate, f.up = st["w"]["g"].data_ptr() + i * E * sg, st["w"]["u"].data_ptr() + i * E * sg
            f.down = st["w"]["d"].data_ptr() + i * E * sd
            f.gate_stride = f.up_stride = sg
            f.down_stride = sd
            fs.append(f)
        nb = KQ.moe_ffn_workspace_bytes(fs[0], B)
        st["ws"] = torch.empty(nb, dtype=torch.uint8, device=DEV)
        st["calls"] = [(ctypes.byref(f), st["xn"].data_ptr() + 4 * i * B * H, st["x"].data_ptr() + 4 * i * B * H, B,
                        st["sel"].data_ptr() + 4 * i * B * k, st["selw"].data_ptr() + 4 * i * B * k, st["ws"].data_ptr(),
                        nb, st["stream"]) for i, f in enumerate(fs)]
        st["keep"] = fs
    return st


def _ok(rc):
    if rc != 0:
        raise RuntimeError(KQ.lib().kq_last_error().decode(errors="replace"))


def run(st):
    kind, L = st["case"]["kind"], st["lib"]
    if kind == "host":
        if L.kq_linear_set_sdot(int(st["case"]["int8"])) < 0:
            raise RuntimeError("kq_linear_set_sdot")
        _ok(L.kq_linear_dispatch(*st["args"]))
        return st["y"]
    if kind == "layer":
        for segs, n in st["calls"]:
            _ok(L.kq_gemv_segments_dev(segs, n, st["stream"]))
        return st["y"]
    if kind == "gemv":
        for a in st["calls"]:
            _ok(L.kq_gemv_dev(*a))
        return st["y"]
    if kind == "multi":
        for a in st["calls"]:
            _ok(st["fn"](*a))
        return st["y"]
    st["x"].copy_(st["res"])          # the residual stream, updated in place by the step
    for a in st["calls"]:
        _ok(L.kq_moe_ffn_dev(*a))
    return {"x": st["x"], "sel": st["sel"], "selw": st["selw"]}


# ------------------------------------------------------------ floor of a pass

def work(case):
    """Weights, inputs and outputs once; two operations per weight and stream."""
    c, kind = case, case["kind"]

    def mat(t, N, K, B=1):
        return N * _row(t, K) + 4 * B * (N + K), 2.0 * N * K * B

    if kind == "host":
        b, f = mat(c["type"], c["N"], c["K"])
    elif kind == "layer":
        H, F = c["H"], c["F"]
        parts = [mat(c["type"], c["Q"] + 2 * c["KV"], H), mat(c["type"], H, c["Q"]), mat(c["type"], 2 * F, H),
                 mat(c["down"], H, F)]
        b, f = c["L"] * (sum(p[0] for p in parts) + 8 * H), c["L"] * sum(p[1] for p in parts)
    elif kind == "gemv":
        b, f = (c["n"] * v for v in mat(c["type"], c["N"], c["K"]))
    elif kind == "multi":
        b, f = (c["n"] * v for v in mat(c["type"], c["N"], c["K"], c["B"]))
    else:
        H, F, E, B, k = c["H"], c["F"], c["E"], c["B"], c["k"]
        distinct = E * (1 - (1 - k / E) ** B)     # expected number of chosen experts
        b = c["L"] * (distinct * (2 * F * _row(c["type"], H) + H * _row(c["down"], F)) + 4 * E * H + 12 * B * H + 8 * B * k)
        f = c["L"] * (2.0 * B * k * 3 * H * F + 2.0 * B * E * H)
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    """Four times what the path shows against 64 bits (sums of 32-bit terms,
    whose order an implementation may choose; the fp16 planes of the mfma mode
    hold 22 bits of x)."""
    if case["kind"] == "moe":
        # near ties may swap experts; in the int8 mode an activation at the
        # middle of two int8 steps may take the other one
        return {"rel": 1.2e-5, "max": 2.5e-4, "differ": 0.001} if case["int8"] else {"rel": 1e-6, "max": 1e-5, "differ": 0.001}
    if case["kind"] == "multi" and case["mode"] == "mfma":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 1.2e-6, "max": 1e-5}


# -------------------------------------------------- the same results, 64 bits

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dq(t, raw, K):
    """Raw block bytes -> [rows, K] weights in float64 (the GGUF definitions)."""
    bb = KQ.BLOCK_BYTES[TYPES[t]]
    b = raw.reshape(-1, bb)
    n = b.shape[0]
    if t in ("Q4_K", "Q5_K"):
        d, dm, s = _f16(b[:, 0:2]), _f16(b[:, 2:4]), b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, bb - 128:].reshape(n, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(n, 8, 32)
        if t == "Q5_K":
            bit = torch.arange(8, device=DEV, dtype=torch.uint8).reshape(1, 8, 1)
            q = q | (((b[:, 16:48].reshape(n, 1, 32) >> bit) & 1) << 4)
        w = (d * sc).reshape(n, 8, 1) * q.double() - (dm * mn).reshape(n, 8, 1)
    elif t == "Q6_K":
        ql, qh, s, d = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32), b[:, 192:208], _f16(b[:, 208:210])
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
        sc = s.contiguous().view(torch.int8).double().reshape(n, 16, 1)
        w = d.reshape(n, 1, 1) * sc * (q.reshape(n, 16, 16).double() - 32)
    elif t == "Q3_K":
        hm, qs, s, d = b[:, :32], b[:, 32:96].reshape(n, 2, 1, 32), b[:, 96:108].to(torch.int32), _f16(b[:, 108:110])
        sh = torch.arange(0, 8, 2, device=DEV, dtype=torch.uint8).reshape(1, 1, 4, 1)
        bit = torch.arange(8, device=DEV, dtype=torch.uint8).reshape(1, 8, 1)
        q = ((qs >> sh) & 3).reshape(n, 8, 32).to(torch.int32)
        q = q - 4 * (1 - ((hm.reshape(n, 1, 32) >> bit) & 1).to(torch.int32))
        lo = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        hi = torch.cat([(s[:, 8:12] >> j) & 3 for j in (0, 2, 4, 6)], 1)
        sc = (lo | (hi << 4)) - 32
        w = (d * sc.double()).reshape(n, 16, 1) * q.reshape(n, 16, 16).double()
    elif t == "Q8_0":
        b = raw.reshape(-1, 34)
        w = _f16(b[:, 0:2]) * b[:, 2:].contiguous().view(torch.int8).double()
    else:
        tail = b[:, 80:84] if t == "Q2_K" else b[:, 144:148]
        d, dm, s = _f16(tail[:, 0:2]), _f16(tail[:, 2:4]), b[:, 0:16]
        if t == "Q2_K":
            sh = torch.arange(0, 8, 2, device=DEV, dtype=torch.uint8).reshape(1, 1, 4, 1)
            q = ((b[:, 16:80].reshape(n, 2, 1, 32) >> sh) & 3).reshape(n, 16, 16)
        else:
            q = b[:, 16:144].reshape(n, 8, 16)
            q = torch.stack([q & 15, q >> 4], 2).reshape(n, 16, 16)
        w = (d * (s & 15).double()).reshape(n, 16, 1) * q.double() - (dm * (s >> 4).double()).reshape(n, 16, 1)
    return w.reshape(-1, K)


def _quantized(x, t):
    """x as the int8 mode sees it: amax/127 per 16 (Q6_K) or 32 values, in binary32."""
    g = x.reshape(*x.shape[:-1], -1, 16 if t == "Q6_K" else 32)
    s = g.abs().amax(-1, keepdim=True)
    s = s / torch.full_like(s, 127.0)      # by a tensor: a scalar divisor becomes a product
    inv = torch.where(s > 0, 1.0 / s, torch.zeros_like(s))
    q = torch.clamp(torch.round(g * inv), -128, 127)
    return (q.double() * s.double()).reshape(x.shape)


def _mul(t, raw, x, K, int8=False):
    """x [B, K] (float32) times the rows of raw, in float64, a few rows at a time."""
    xd = _quantized(x, t) if int8 and t in INT8 else x.double()
    rb, out = _row(t, K), []
    rows = len(raw) // rb
    step = max(1, (1 << 26) // K)
    for r in range(0, rows, step):
        out.append(xd @ _dq(t, raw[r * rb:min(rows, r + step) * rb], K).t().contiguous())
    return torch.cat(out, -1)


def exact(case, seed):
    c, kind = dict(case), case["kind"]
    if kind == "host":
        w = _weights(7, 0, c["type"], c["N"], c["K"])
        return _mul(c["type"], w, _x(seed, 1, c["K"]).reshape(1, -1), c["K"], c["int8"]).reshape(-1).cpu().numpy()
    if kind == "layer":
        H, Q, KV, F, n, t, td = c["H"], c["Q"], c["KV"], c["F"], c["L"], c["type"], c["down"]
        out = {}
        for name, salt, xs, tt, N, K, add in (("qkv", 1, 5, t, Q + 2 * KV, H, False), ("o", 2, 6, t, H, Q, True),
                                              ("gu", 3, 7, t, 2 * F, H, False), ("d", 4, 8, td, H, F, True)):
            w, x, r = _weights(seed, salt, tt, n * N, K).reshape(n, -1), _x(seed, xs, n, K), _x(seed, 9, n, H)
            out[name] = torch.stack([_mul(tt, w[i], x[i:i + 1], K, c["int8"])[0] + (r[i].double() if add else 0)
                                     for i in range(n)])
        return out
    if kind == "gemv":
        n, N, K, t = c["n"], c["N"], c["K"], c["type"]
        w, x = _weights(seed, 1, t, n * N, K).reshape(n, -1), _x(seed, 2, n, K)
        return torch.stack([_mul(t, w[i], x[i:i + 1], K, c["int8"])[0] for i in range(n)])
    if kind == "multi":
        n, N, K, t, B = c["n"], c["N"], c["K"], c["type"], c["B"]
        w, x = _weights(seed, 1, t, n * N, K).reshape(n, -1), _x(seed, 2, B, K)
        return torch.stack([_mul(t, w[i], x, K, c["mode"] == "int8") for i in range(n)])
    H, F, E, B, n, k, t, td = (c[v] for v in ("H", "F", "E", "B", "L", "k", "type", "down"))
    wg, wu = (_weights(seed, s, t, n * E * F, H).reshape(n, E, -1) for s in (1, 2))
    wd = _weights(seed, 3, td, n * E * H, F).reshape(n, E, -1)
    router, xn, x = _x(seed, 4, n, E, H) * 0.03, _x(seed, 5, n, B, H), _x(seed, 6, n, B, H).double()
    sel, selw = torch.empty(n, B, k, dtype=torch.int32, device=DEV), torch.empty(n, B, k, device=DEV, dtype=torch.float64)
    for i in range(n):
        p = torch.softmax(xn[i].double() @ router[i].double().t().contiguous(), -1)
        v, s = torch.sort(p, dim=-1, descending=True, stable=True)
        sel[i], selw[i] = s[:, :k].int(), v[:, :k]
        for e in torch.unique(sel[i]).tolist():
            b, r = torch.nonzero(sel[i] == e, as_tuple=True)
            a = xn[i][b]
            g, u = _mul(t, wg[i, e], a, H, c["int8"]), _mul(t, wu[i, e], a, H, c["int8"])
            act = g / (1 + torch.exp(-g)) * u
            # the int8 mode quantizes the binary32 activations
            o = _mul(td, wd[i, e], act.float(), F, True) if c["int8"] else act @ _dq(td, wd[i, e], F).t().contiguous()
            x[i].index_add_(0, b, o * selw[i][b, r].unsqueeze(1))
    return {"x": x, "sel": None, "selw": selw}
