"""Workloads that callers of libkv-compact.so run, as measured cases.

Each case is one whole call through a public entry point, with what the caller
holds before it: a KV cache (resident in HBM for the device entries, host
arrays for the drop-in entry), the parameters and the result buffers.

Shapes are those of this repository's benchmark, its full-size tests and the
reference's published tables: Llama-3-8B-like caches (32 layers x 8 KV heads x
128), long bfloat16 caches with 256-wide heads, Q8_0 / Q4_0 caches, llama.cpp
sequence states, single layers and single heads. Keys are N(0, 1) times a
per-channel LogNormal(0, 0.5) scale, values N(0, 1), SnapKV reference queries
the last keys plus N(0, 0.1^2) noise; "n_q": 0 stands for the library's own
cheap reference queries.

The library returns the reference's fp32 results bit for bit, so every output
is compared exactly.
"""
from __future__ import annotations

import ctypes
import math
import struct
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "kv-compact_amd"))

import kvcompact as kc  # noqa: E402

F16, Q4_0, Q8_0, BF16 = kc.KV_TYPE_F16, kc.KV_TYPE_Q4_0, kc.KV_TYPE_Q8_0, kc.KV_TYPE_BF16
TYPES = {"f16": F16, "q4_0": Q4_0, "q8_0": Q8_0, "bf16": BF16}

_lib = None


def _library():
    global _lib
    if _lib is None:
        _lib = kc.load_product()
        kc.bind_device_api(_lib.dll)
        f = _lib.dll.kvc_state_compact_device
        f.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.POINTER(kc.StateParams), ctypes.c_void_p,
                      ctypes.c_size_t, ctypes.POINTER(ctypes.c_size_t), ctypes.c_void_p, ctypes.c_void_p]
        f.restype = ctypes.c_int
    return _lib


# ------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest call: one layer of a short prompt (the first size of the
        # reference's quantized bench), where launches and waits count
        dict(name="one_layer_256", entry="layers", L=1, T=256, H=4, d=64, n_q=0, ratio=0.5),
        # one attention head of one layer, 4 outlier channels, half kept
        dict(name="one_head_4096", entry="layers", L=1, T=4096, H=1, d=128, n_q=0, ratio=0.5, outliers=4),
        # a Llama-3-8B-shaped cache of an ordinary context, diverse selection
        dict(name="llama_16k_diverse", entry="layers", L=32, T=16384, H=8, d=128, n_q=32, ratio=0.2, diversity=1),
        # the largest: the same cache at 100k tokens (the benchmark's workload)
        dict(name="llama_100k_diverse", entry="layers", L=32, T=100000, H=8, d=128, n_q=32, ratio=0.2, diversity=1),
        # a few layers of narrow heads (the reference's auto-chunk bench shape)
        # with the attention-bias fit, clamped least squares
        dict(name="bias_fit_10240", entry="layers", L=4, T=10240, H=4, d=64, n_q=0, ratio=0.5, beta="ls"),
        # everything on: Lawson-Hanson bias fit, diverse selection, one
        # refinement round, 30% of the tokens down-weighted as thinking
        dict(name="full_options_20011", entry="layers", L=10, T=20011, H=4, d=128, n_q=32, ratio=0.2, diversity=1,
             beta="lh", refine=1, thinking=0.3),
        # long bfloat16 cache of hybrid-attention layers with 256-wide heads
        dict(name="bf16_100k_d256", entry="quantized", type="bf16", L=10, T=100000, H=4, d=256, n_q=32, ratio=0.5),
        # quantized caches of a 32-layer model: 32k tokens, and a short ragged one
        dict(name="q8_0_32k", entry="quantized", type="q8_0", L=32, T=32768, H=8, d=128, n_q=0, ratio=0.2),
        dict(name="q4_0_3001", entry="quantized", type="q4_0", L=32, T=3001, H=8, d=128, n_q=32, ratio=0.2),
        # llama.cpp sequence states: F16 rows of a 2048-cell context, and a
        # short ragged Q8_0 one of a few layers with F16 values stored transposed
        dict(name="state_f16_2048", entry="state", type="f16", v_trans=0, L=32, T=2048, H=8, d=128, ratio=0.2),
        dict(name="state_q8_777", entry="state", type="q8_0", v_trans=1, L=8, T=777, H=4, d=64, ratio=0.3),
        # the drop-in call on host memory, one layer of an ordinary context
        dict(name="host_layer_16k", entry="host", L=1, T=16384, H=8, d=128, n_q=32, ratio=0.2),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    entry = rng.choice(["layers", "layers", "layers", "options", "quantized", "quantized", "state", "host"])
    while True:
        if entry == "state":
            c = dict(entry="state", type=rng.choice(["f16", "q8_0"]), v_trans=rng.choice([0, 1]), L=_log(rng, 1, 32),
                     T=_log(rng, 128, 4096), H=rng.choice([2, 4, 8]), d=rng.choice([64, 128]),
                     ratio=rng.choice([0.1, 0.2, 0.3, 0.5]))
            if c["L"] * c["H"] * (c["T"] * c["ratio"]) ** 3 > 256 * 409.0 ** 3:
                continue
            return c
        c = dict(entry=entry, L=_log(rng, 1, 32), T=_log(rng, 64, 100000), H=rng.choice([1, 2, 4, 8]),
                 d=rng.choice([32, 64, 96, 128, 256]), n_q=rng.choice([0, 0, 16, 32, 64]),
                 ratio=rng.choice([0.1, 0.2, 0.2, 0.3, 0.5, 0.5, 0.8]))
        if entry == "host":
            c.update(L=1, T=_log(rng, 256, 32768))
        elif entry == "quantized":
            c["type"] = rng.choice(["q8_0", "q4_0", "bf16", "f16"])
        else:
            if c["ratio"] >= 0.2 and rng.random() < 0.5:
                c["diversity"] = 1
            if entry == "options":
                c.update(entry="layers", L=min(c["L"], 10), T=min(c["T"], 25000), H=min(c["H"], 4),
                         beta=rng.choice(["ls", "ls", "lh"]))
                if rng.random() < 0.5:
                    c["refine"] = 1
                if rng.random() < 0.5:
                    c["thinking"] = 0.3
        c["n_q"] = min(c["n_q"], c["T"])
        heads = c["L"] * c["T"] * c["H"]
        if heads * c["d"] > 32 * 100000 * 1024 // 2 or heads * c["ratio"] > 32 * 100000 * 8 * 0.2 / 2:
            continue
        return c


# ------------------------------------------------------------------ inputs

def _params(c):
    lib = _library()
    p = lib.params(target_ratio=c["ratio"], use_diversity=c.get("diversity", 0), use_cheap_qref=0 if c["n_q"] else 1,
                   refine_rounds=c.get("refine", 0))
    if c.get("beta"):
        p.skip_beta = 0
        p.nnls_method = 0 if c["beta"] == "lh" else 1
    return p


def _keys_values(c, gen):
    """K, V fp32 [L][T][H * d] and the SnapKV queries [L][n_q][H * d] (or None)."""
    L, T, E, n_q = c["L"], c["T"], c["H"] * c["d"], c.get("n_q", 0)
    K = torch.empty(L, T, E, device="cuda")
    V = torch.empty(L, T, E, device="cuda")
    Q = torch.empty(L, n_q, E, device="cuda") if n_q else None
    for l in range(L):
        K[l].normal_(generator=gen)
        V[l].normal_(generator=gen)
        if c.get("outliers"):
            ch = torch.randperm(E, generator=gen, device="cuda")[:c["outliers"]]
            K[l][:, ch] *= 8.0
            V[l][:, ch] *= 8.0
        else:
            K[l] *= torch.exp(0.5 * torch.randn(E, generator=gen, device="cuda"))
        if n_q:
            Q[l] = K[l, T - n_q:] + 0.1 * torch.randn(n_q, E, generator=gen, device="cuda")
    return K, V, Q


def _encode(x, typ):
    """fp32 rows [..., n] -> uint8 rows of the codec."""
    if typ == F16:
        return x.half().view(torch.uint8)
    if typ == BF16:
        return x.bfloat16().view(torch.uint8)
    b = x.unflatten(-1, (-1, 32))
    lim = 127.0 if typ == Q8_0 else 7.0
    d = b.abs().amax(-1, keepdim=True) / lim
    q = torch.round(b / d.clamp_min(1e-30)).clamp_(-lim, lim)
    if typ == Q8_0:
        codes = q.to(torch.int8).view(torch.uint8)
    else:
        u = (q + 8.0).to(torch.uint8)
        codes = u[..., 0::2] | (u[..., 1::2] << 4)
    return torch.cat([d.half().view(torch.uint8), codes], -1).flatten(-2)


def _row_bytes(typ, n):
    return {F16: 2 * n, BF16: 2 * n, Q8_0: n // 32 * 34, Q4_0: n // 32 * 18}[typ]


def _outputs(L, t, H, d):
    """Result buffers; the statistics' columns are named views of one [L][3] array."""
    stats = torch.zeros(L, 3, device="cuda")
    return stats, dict(indices=torch.zeros(L, t, dtype=torch.int32, device="cuda"),
                       beta=torch.zeros(L, H, t, device="cuda"), C_v=torch.zeros(L, H, t, d, device="cuda"),
                       avg_cosine_sim=stats[:, 0], avg_mse=stats[:, 1], avg_agreement=stats[:, 2])


def _blob(c, gen):
    """A llama.cpp sequence state in device memory: one stream, one sequence id per cell."""
    L, T, E, typ = c["L"], c["T"], c["H"] * c["d"], TYPES[c["type"]]
    cells = np.zeros(T, dtype=[("pos", "<i4"), ("n", "<u4"), ("seq", "<i4")])
    cells["pos"] = np.arange(T)
    cells["n"] = 1

    def raw(b):
        return torch.frombuffer(bytearray(b), dtype=torch.uint8).cuda()

    K, V, _ = _keys_values(c, gen)
    parts = [raw(struct.pack("<II", 1, T) + cells.tobytes() + struct.pack("<II", c["v_trans"], L))]
    for l in range(L):
        rows = _encode(K[l], typ)
        parts += [raw(struct.pack("<iQ", typ, rows.shape[1])), rows.reshape(-1)]
    for l in range(L):
        if c["v_trans"]:   # [channel][cell], as stored without flash attention
            parts += [raw(struct.pack("<iII", F16, 2, E)), V[l].t().contiguous().half().view(torch.uint8).reshape(-1)]
        else:
            rows = _encode(V[l], typ)
            parts += [raw(struct.pack("<iQ", typ, rows.shape[1])), rows.reshape(-1)]
    return torch.cat(parts)


def prepare(case, seed):
    lib = _library()
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if c["entry"] == "state":
        blob = _blob(c, gen)
        p, keep = kc.state_params(c["ratio"], c["H"])
        t = max(1, int(np.float32(c["T"]) * np.float32(c["ratio"])))
        s = dict(case=c, blob=blob, params=p, keep=keep, out=torch.zeros_like(blob), selected=np.zeros(t, np.int32))
        torch.cuda.synchronize()
        return s
    p = _params(c)
    K, V, Q = _keys_values(c, gen)
    s = dict(case=c, params=p, Q=Q)
    if c["entry"] == "host":
        s.update(K=K[0].cpu().numpy(), V=V[0].cpu().numpy(), Q=Q[0].cpu().numpy() if Q is not None else None)
        return s
    L, T, H, d = c["L"], c["T"], c["H"], c["d"]
    t, _ = kc.plan(lib.dll, T, c["n_q"], Q is not None, p)
    s["stats"], s["out"] = _outputs(L, t, H, d)
    if c["entry"] == "quantized":
        typ = TYPES[c["type"]]
        s["K"] = torch.stack([_encode(K[l], typ) for l in range(L)])
        s["V"] = torch.stack([_encode(V[l], typ) for l in range(L)])
        rb = _row_bytes(typ, H * d)
        s["out"].update(K_out=torch.zeros(L, t, rb, dtype=torch.uint8, device="cuda"),
                        V_out=torch.zeros(L, t, rb, dtype=torch.uint8, device="cuda"))
    else:
        s.update(K=K, V=V, weights=None)
        if c.get("thinking"):
            n = max(1, int(T * c["thinking"]))
            at = int(torch.randint(0, T - n + 1, (1,), generator=gen, device="cuda"))
            s["weights"] = torch.ones(T, device="cuda")
            s["weights"][at:at + n] = 0.5
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- run

def _check(rc, what):
    if rc != 0:
        raise RuntimeError(f"{what} returned {rc}")


def run(state):
    lib = _library()
    dll = lib.dll
    s, c = state, state["case"]
    L, T, H, d = c["L"], c["T"], c["H"], c["d"]
    E = H * d
    if c["entry"] == "state":
        n = ctypes.c_size_t(0)
        _check(dll.kvc_state_compact_device(s["blob"].data_ptr(), s["blob"].numel(), ctypes.byref(s["params"]),
                                            s["out"].data_ptr(), s["out"].numel(), ctypes.byref(n),
                                            s["selected"].ctypes.data, None), "kvc_state_compact_device")
        return dict(blob=s["out"][:n.value], selected=s["selected"])
    if c["entry"] == "host":
        r = lib.compact(s["K"], s["V"], s["Q"], T, c["n_q"], H, d, d, s["params"])
        return dict(indices=r.indices, beta=r.beta, C_v=r.C_v,
                    stats=[r.stats["avg_cosine_sim"], r.stats["avg_mse"], r.stats["avg_agreement"]])
    o = s["out"]
    dev = kc.DeviceOut(o["indices"].data_ptr(), o["beta"].data_ptr(), o["C_v"].data_ptr(),
                       s["stats"].data_ptr())
    q = s["Q"].data_ptr() if s["Q"] is not None else None
    if c["entry"] == "quantized":
        typ = TYPES[c["type"]]
        rb = _row_bytes(typ, E)
        _check(dll.kvc_compact_quantized_layers_device(
            s["K"].data_ptr(), s["V"].data_ptr(), q, L, typ, typ, rb, rb, T, c["n_q"], H, d, d, T * rb, T * rb,
            c["n_q"] * E, ctypes.byref(s["params"]), ctypes.byref(dev), o["K_out"].data_ptr(), o["V_out"].data_ptr(),
            None), "kvc_compact_quantized_layers_device")
        return o
    w = s["weights"].data_ptr() if s["weights"] is not None else None
    _check(dll.kvc_compact_layers_device(
        s["K"].data_ptr(), s["V"].data_ptr(), q, L, T, c["n_q"], H, d, d, T * E, T * E, c["n_q"] * E,
        ctypes.byref(s["params"]), w, ctypes.byref(dev), None), "kvc_compact_layers_device")
    return o


# -------------------------------------------------------------------- work

def _chunk_plan(c):
    """[(start, keys, kept)] of one layer: the library's automatic plan in the same fp32 steps."""
    T, r = c["T"], np.float32(c["ratio"])
    if c["entry"] == "state":
        return [(0, T, max(1, int(np.float32(T) * r)))]
    est = int(np.float32(T) * r)
    cs = min(T, max(64, int(np.float32(256.0) / r))) if est > 256 else T
    return [(a, min(cs, T - a), min(min(cs, T - a), max(1, int(np.float32(min(cs, T - a)) * r))))
            for a in range(0, T, cs)]


def _cheap(n):
    return min(n, max(4, min(64, n // 2)))


def work(case):
    c = case
    L, T, H, d = c["L"], c["T"], c["H"], c["d"]
    E, units = H * d, L * H
    plan = _chunk_plan(c)
    kept = sum(t for _, _, t in plan)
    flops = 0.0
    for _, n, t in plan:
        nq = max(16, T // 4) if c["entry"] == "state" else c["n_q"] or _cheap(n)
        rhs = d
        # scores, refit target, Gram matrix and right-hand sides, elimination, substitution
        f = 4.0 * nq * n * d + 1.0 * nq * t * (t + 1) + 2.0 * nq * t * rhs + 2.0 / 3 * t ** 3 + 2.0 * t * t * rhs
        if c.get("beta"):
            f += 1.0 * nq * t * (t + 1) + 2.0 / 3 * t ** 3
        flops += units * f
        if c.get("diversity"):
            flops += L * 1.0 * t * t * E   # cosines between the kept keys at the least
    if c["entry"] == "state":
        typ = TYPES[c["type"]]
        row = _row_bytes(typ, E) + (2 * E if c["v_trans"] else _row_bytes(typ, E)) + 12.0 / L
        return dict(bytes=L * row * (T + kept), flops=flops)
    out = L * kept * (4 + 4 * H + 4 * E)
    if c["entry"] == "quantized":
        rb = _row_bytes(TYPES[c["type"]], E)
        return dict(bytes=2.0 * L * rb * (T + kept) + 4.0 * L * c["n_q"] * E + out, flops=flops)
    return dict(bytes=8.0 * L * T * E + 4.0 * L * c["n_q"] * E + out, flops=flops)


def tolerance(case):
    # The documented contract: indices, biases, values, statistics and encoded
    # rows equal the reference's fp32 results bit for bit. (A refitted value
    # has no looser bound that means anything: with more kept keys than
    # reference queries the least squares are underdetermined, and rounding
    # alone moves single values by percents.)
    return "exact"


# ------------------------------------------------- 64-bit results for checking

def _decode(rows, typ):
    if typ == F16:
        return rows.view(torch.float16).double()
    if typ == BF16:
        return rows.view(torch.bfloat16).double()
    b = rows.unflatten(-1, (-1, 34 if typ == Q8_0 else 18))
    d = b[..., :2].contiguous().view(torch.float16).double()
    if typ == Q8_0:
        q = b[..., 2:].contiguous().view(torch.int8).double()
    else:
        n = b[..., 2:]
        q = torch.stack([n & 15, n >> 4], -1).flatten(-2).double() - 8.0
    return (q * d).flatten(-2)


def _sample(n, T):
    """The library's reference-query positions over T keys (its fp32 arithmetic)."""
    f = (np.arange(1, n + 1, dtype=np.float32) / np.float32(n + 1)) ** 2
    return torch.from_numpy(np.clip((f * np.float32(T - 1)).astype(np.int64), 0, T - 1)).cuda()


def exact(case, seed):
    # Single kept values, and the mean squared error that hangs on them, have
    # no 64-bit counterpart (underdetermined least squares, see tolerance());
    # the cosine between full and compacted attention outputs has one. Options
    # that select or fit step by step, blobs, and the larger caches are left to
    # the exact comparison, and so are chunks that each fit their own sampled
    # queries: the statistics then ask them about other queries, where the
    # underdetermined fits' fp32 rounding shows (percents of the cosine).
    c = case
    if not c.get("n_q") and len(_chunk_plan(c)) > 1:
        return None
    L, T, H, d = c["L"], c["T"], c["H"], c["d"]
    if (c["entry"] not in ("layers", "quantized") or c.get("diversity") or c.get("beta") or c.get("refine") or
            c.get("thinking") or L * T * H * d > 32 * 4000 * 1024):
        return None
    s = prepare(c, seed)
    cos = []
    for l in range(L):
        K, V = (_decode(s[n][l], TYPES[c["type"]]) if c["entry"] == "quantized" else s[n][l].double() for n in "KV")
        K, V = (x.view(T, H, d).transpose(0, 1).contiguous() for x in (K, V))   # [H][T][d]
        given = s["Q"][l].double().view(-1, H, d).transpose(0, 1).contiguous() if c["n_q"] else None

        def scores(q, k):
            return q @ k.transpose(1, 2).contiguous() / math.sqrt(d)

        hs = min(H, 4)
        Qs = given if given is not None else K[:, _sample(_cheap(T), T)]
        Qs = Qs[:hs, :32].contiguous()
        full = torch.softmax(scores(Qs, K[:hs]), -1) @ V[:hs]
        plan = _chunk_plan(c)
        num, den = [], []
        for start, n, t in plan:
            k, v = K[:, start:start + n].contiguous(), V[:, start:start + n].contiguous()
            q = given if given is not None else k[:, _sample(_cheap(n), n)].contiguous()
            S = scores(q, k)
            A = torch.softmax(S, -1)
            keep = A.square().mean(1).sqrt().amax(0).topk(t).indices.sort().values
            X = torch.softmax(S[:, :, keep], -1)
            ridge = 1e-6 * torch.eye(X.shape[1], dtype=torch.float64, device="cuda")
            # (X'X + r I)^-1 X' Y in its dual form
            C = X.transpose(1, 2).contiguous() @ torch.linalg.solve(X @ X.transpose(1, 2).contiguous() + ridge, A @ v)
            e = scores(Qs, k[:hs, keep].contiguous())
            num.append((e, C[:hs].contiguous()))
            den.append(e)
        P = torch.softmax(torch.cat(den, -1), -1)
        out, at = torch.zeros_like(full), 0
        for e, C in num:
            out += P[:, :, at:at + e.shape[2]].contiguous() @ C
            at += e.shape[2]
        norm = full.norm(dim=-1) * out.norm(dim=-1) + 1e-8
        cos.append(((full * out).sum(-1) / norm).mean())
    r = {k: None for k in s["out"]}
    r["avg_cosine_sim"] = torch.stack(cos)
    return r
