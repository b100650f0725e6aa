"""The work that a user of this backend has it do, for timing and for comparing two builds.

Every case goes through the Python operators of yllm_amd (attention.py, gdn.py), eagerly, on torch's
current stream, with the workspaces, weights, caches and output rows that an engine keeps.  Kinds:

  token    one decode token of an attention layer after its projections: RoPE + KV store + decode in
           one call, then o_proj and the residual add
  block    the same layer over T prompt tokens: RoPE + KV store, causal prefill, o_proj; fp32 rows
           throughout, as the engine holds them
  decode   attention of one token over a long cache
  batch    one token each of several independent sequences of different lengths
  prefill  causal attention over T prompt tokens whose keys are stored, 16-bit queries and outputs,
           with the qwen35 sigmoid gate where `gated`
  gdn      a Gated-DeltaNet layer over T prompt tokens after its projections: gates, conv + silu,
           recurrence, gated RMSNorm
  hybrid   one decode token of the qwen35 group: three Gated-DeltaNet layers and a gated attention layer
  rope     RoPE + KV store of T prompt tokens, 16-bit queries out (the step ahead of `prefill`)
  oproj    o_proj of T tokens from 16-bit attention outputs (the step after `prefill`)
"""
from __future__ import annotations

import math

import torch

from yllm_amd import attention as A
from yllm_amd import gdn as G

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ROPES = {"pairs": A.ROPE_PAIRS, "half": A.ROPE_HALF, "mrope": A.ROPE_MROPE}
# (query heads, kv heads, head_dim, rope, theta): the head layouts of the benchmark's configurations
HEADS = [(14, 2, 64, "half", 1e6), (28, 4, 128, "half", 1e6), (32, 8, 128, "pairs", 5e5)]
KW = 4  # conv taps of a Gated-DeltaNet layer
N_ROT = 64  # rotated dimensions of a qwen35 head


def _h(i: int) -> dict:
    nh, nkv, d, rope, theta = HEADS[i]
    return {"nh": nh, "nkv": nkv, "d": d, "rope": rope, "theta": theta}


QWEN35 = {"nh": 16, "nkv": 2, "d": 256, "rope": "mrope", "theta": 1e7}


def listed() -> list[dict]:
    return [
        # the smallest call: one token of the reference's CPU-runnable model, 512 keys
        {"name": "token_512", "kind": "token", **_h(0), "pos": 511},
        # a decode step of the qwen35 group after a 4096-token prompt: a chain of short launches
        {"name": "hybrid_token_4k", "kind": "hybrid", **QWEN35, "pos": 4223, "gh": 16, "gd": 128},
        # decode deep into one long context: a single stream over the cache
        {"name": "decode_32k", "kind": "decode", **_h(2), "keys": 32768},
        # serving: 64 sequences, ragged between 1k and 32k keys
        {"name": "batch_64", "kind": "batch", **_h(2), "n_seq": 64, "lo": 1024, "hi": 32768},
        # the engine's own prefill call: 64 tokens against the prefix stored so far
        {"name": "block_64_at_1984", "kind": "block", **_h(1), "T": 64, "start": 1984},
        # a whole 2048-token prompt in one call, fp32 rows as the engine holds them
        {"name": "block_2k", "kind": "block", **_h(1), "T": 2048, "start": 0},
        # a long prompt, 16-bit queries and outputs
        {"name": "prefill_8k", "kind": "prefill", **_h(2), "T": 8192, "start": 0, "dtype": "f16", "gated": False},
        # the qwen35 gated attention over its 4096-token prompt
        {"name": "gated_4k", "kind": "prefill", **QWEN35, "T": 4096, "start": 0, "dtype": "bf16", "gated": True},
        # a Gated-DeltaNet layer in the engine's 64-token calls, and over the whole prompt
        {"name": "gdn_64", "kind": "gdn", "T": 64, "gh": 16, "gd": 128},
        {"name": "gdn_4k", "kind": "gdn", "T": 4096, "gh": 16, "gd": 128},
        # the steps around a long prompt's attention
        {"name": "rope_8k", "kind": "rope", **_h(2), "T": 8192, "start": 0, "dtype": "f16"},
        {"name": "oproj_8k", "kind": "oproj", "T": 8192, "hidden": 4096, "qdim": 4096},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng) -> dict:
    kind = rng.choice(["token", "block", "block", "decode", "batch", "prefill", "prefill", "gdn", "gdn", "hybrid",
                       "rope", "oproj"])
    h = _h(rng.randrange(len(HEADS)))
    if kind == "token":
        return {"kind": kind, **h, "pos": _log(rng, 1, 16384) - 1}
    if kind == "block":
        return {"kind": kind, **h, "T": _log(rng, 2, 2048), "start": rng.choice([0, _log(rng, 1, 4096)])}
    if kind == "decode":
        return {"kind": kind, **h, "keys": _log(rng, 256, 131072)}
    if kind == "batch":
        hi = _log(rng, 1024, 32768)
        return {"kind": kind, **h, "n_seq": _log(rng, 2, 48), "lo": max(1, hi // 32), "hi": hi}
    if kind == "prefill":
        if rng.random() < 0.4:
            return {"kind": kind, **QWEN35, "T": _log(rng, 100, 4096), "start": 0, "dtype": "bf16", "gated": True}
        return {"kind": kind, **h, "T": _log(rng, 100, 6144), "start": rng.choice([0, 0, _log(rng, 64, 2048)]),
                "dtype": rng.choice(["f16", "bf16"]), "gated": False}
    if kind == "gdn":
        return {"kind": kind, "T": _log(rng, 64, 4096), "gh": rng.choice([16, 16, 32]), "gd": rng.choice([64, 128, 128])}
    if kind == "hybrid":
        return {"kind": kind, **QWEN35, "pos": _log(rng, 64, 16384), "gh": rng.choice([16, 16, 32]), "gd": 128}
    if kind == "rope":
        h = rng.choice([h, h, QWEN35])
        return {"kind": kind, **h, "T": _log(rng, 100, 8192), "start": rng.choice([0, _log(rng, 1, 4096)]),
                "dtype": rng.choice(["f16", "bf16"])}
    qdim = rng.choice([896, 3584, 4096])
    return {"kind": "oproj", "T": _log(rng, 1, 8192), "hidden": qdim, "qdim": qdim}


# ---- inputs ------------------------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, scale: float = 1.0) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _cache(g, c: dict, rows: int, capacity: int) -> A.LayerKV:
    """A layer cache whose first `rows` positions hold keys and values."""
    cache = A.LayerKV.empty(c["nkv"], c["d"], capacity)
    if rows:
        kvd = c["nkv"] * c["d"]
        A.kv_store(cache, _normal(g, rows, kvd).half(), _normal(g, rows, kvd, scale=0.5).half(), 0)
    return cache


def _lens(c: dict, seed: int) -> list[int]:
    g = torch.Generator().manual_seed(int(seed))
    return torch.randint(c["lo"], c["hi"] + 1, (c["n_seq"],), generator=g).tolist()


def _gdn_weights(g, gh: int, gd: int) -> dict:
    conv = 3 * gh * gd
    return {"conv_w": _normal(g, conv, KW, scale=0.5),
            "dt_bias": _normal(g, gh, scale=0.5),
            "ssm_a": -torch.exp(torch.rand(gh, generator=g, device="cuda") * 2.0 - 1.0),
            "norm_w": 1.0 + _normal(g, gd, scale=0.1)}


def _gdn_state(g, gh: int, gd: int) -> dict:
    conv = 3 * gh * gd
    S = _normal(g, gh, gd, gd, scale=0.05)
    line = _normal(g, KW, conv, scale=0.5)
    return {"S": S, "S2": torch.empty_like(S), "line": line, "line2": torch.empty_like(line)}


def prepare(case: dict, seed: int) -> dict:
    c, g, kind = case, _gen(seed), case["kind"]
    s = {"c": c}
    if kind in ("token", "block", "decode", "batch", "prefill", "hybrid", "rope"):
        nh, nkv, d = c["nh"], c["nkv"], c["d"]
        qd, kvd = nh * d, nkv * d
    if kind == "token":
        n = c["pos"] + 1
        s["cache"] = _cache(g, c, c["pos"], n)
        s["qkv"] = _normal(g, qd + 2 * kvd)
        s["ws"] = A.decode_workspace(A.decode_workspace_bytes(1, n, n, nh, nkv, d))
        s["att"] = torch.empty(qd, device="cuda")
        s["w"] = _normal(g, qd, qd, scale=qd ** -0.5).half()
        s["x"] = _normal(g, qd)
    elif kind == "block":
        T, end = c["T"], c["start"] + c["T"]
        s["cache"] = _cache(g, c, c["start"], end)
        s["qkv"] = _normal(g, T, qd + 2 * kvd)
        s["q"] = torch.empty((T, qd), device="cuda")
        s["ws"] = A.prefill_workspace(A.prefill_workspace_bytes(T, end, nh, nkv, d))
        s["att"] = torch.empty((T, qd), device="cuda")
        s["w"] = _normal(g, qd, qd, scale=qd ** -0.5).half()
        s["x"] = _normal(g, T, qd)
        s["ows"] = torch.empty(max(256, A.o_proj_workspace_bytes(T, qd, qd, torch.float16)), dtype=torch.uint8,
                               device="cuda")
    elif kind == "decode":
        n = c["keys"]
        s["cache"] = _cache(g, c, n, n)
        s["q"] = _normal(g, qd)
        s["ws"] = A.decode_workspace(A.decode_workspace_bytes(1, n, n, nh, nkv, d))
        s["att"] = torch.empty(qd, device="cuda")
    elif kind == "batch":
        s["lens"] = lens = _lens(c, seed)
        s["batch"] = A.DecodeBatch([_cache(g, c, n, c["hi"]) for n in lens])
        s["lens_dev"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
        s["q"] = _normal(g, len(lens), qd)
        s["ws"] = A.decode_workspace(A.decode_workspace_bytes(len(lens), max(lens), sum(lens), nh, nkv, d))
        s["att"] = torch.empty((len(lens), qd), device="cuda")
    elif kind == "prefill":
        T, end, dt = c["T"], c["start"] + c["T"], DTYPES[c["dtype"]]
        s["cache"] = _cache(g, c, end, end)
        s["q"] = _normal(g, T, qd).to(dt)
        s["gate"] = _normal(g, T, qd) if c["gated"] else None
        s["ws"] = A.prefill_workspace(A.prefill_workspace_bytes(T, end, nh, nkv, d))
        s["att"] = torch.empty((T, qd), dtype=dt, device="cuda")
    elif kind == "gdn":
        T, gh, gd = c["T"], c["gh"], c["gd"]
        s.update(_gdn_weights(g, gh, gd), **_gdn_state(g, gh, gd))
        s["qkv"] = _normal(g, T, 3 * gh * gd)
        s["z"] = _normal(g, T, gh * gd)
        s["alpha"], s["beta"] = _normal(g, T, gh), _normal(g, T, gh)
        s["gate"] = torch.empty((T, gh), device="cuda")
        s["rows"] = torch.empty((T, 3 * gh * gd), device="cuda")
        s["out"] = torch.empty((T, gh * gd), device="cuda")
        s["ws"] = torch.empty(max(64, G.gdn_chunk_workspace_bytes(T, gh, gd) // 4), device="cuda")
    elif kind == "hybrid":
        n, gh, gd = c["pos"] + 1, c["gh"], c["gd"]
        s["layers"] = [dict(_gdn_weights(g, gh, gd), **_gdn_state(g, gh, gd), qkv=_normal(g, 3 * gh * gd),
                            z=_normal(g, gh * gd), alpha=_normal(g, gh), beta=_normal(g, gh),
                            y=torch.empty(gh * gd, device="cuda")) for _ in range(3)]
        s["cache"] = _cache(g, c, c["pos"], n)
        s["qkv"] = _normal(g, qd + 2 * kvd)
        s["gate"] = _normal(g, qd)
        s["ws"] = A.decode_workspace(A.decode_workspace_bytes(1, n, n, nh, nkv, d))
        s["att"] = torch.empty(qd, device="cuda")
    elif kind == "rope":
        T, end = c["T"], c["start"] + c["T"]
        s["cache"] = A.LayerKV.empty(nkv, d, end)
        s["qkv"] = _normal(g, T, qd + 2 * kvd)
        s["q"] = torch.empty((T, qd), dtype=DTYPES[c["dtype"]], device="cuda")
    elif kind == "oproj":
        T, hidden, qdim = c["T"], c["hidden"], c["qdim"]
        s["att"] = _normal(g, T, qdim, scale=0.5).half()
        s["w"] = _normal(g, hidden, qdim, scale=qdim ** -0.5).half()
        s["x"] = _normal(g, T, hidden)
    return s


# ---- one pass ----------------------------------------------------------------------------------

def _rope_args(c: dict) -> tuple:
    return ROPES[c["rope"]], c["theta"], N_ROT if c["rope"] == "mrope" else 0


def _split(s: dict, c: dict) -> tuple:
    """q, k and v of the fused projection row(s)."""
    qd, kvd, x = c["nh"] * c["d"], c["nkv"] * c["d"], s["qkv"]
    return x[..., :qd], x[..., qd:qd + kvd], x[..., qd + kvd:]


def run(s: dict):
    c = s["c"]
    kind = c["kind"]
    if kind == "token":
        # x is the residual stream: o_proj adds to it in place (another pass adds once more)
        q, k, v = _split(s, c)
        rope, theta, n_rot = _rope_args(c)
        A.attn_decode_rope(q, k, v, s["cache"], c["pos"], c["nh"], rope, theta, n_rot, out=s["att"],
                           workspace=s["ws"])
        A.o_proj(s["x"], s["att"], s["w"])
        return s["att"], s["x"], s["cache"].k, s["cache"].v
    if kind == "block":
        q, k, v = _split(s, c)
        rope, theta, n_rot = _rope_args(c)
        A.rope_kv_store(s["cache"], q, k, v, c["start"], c["nh"], rope, theta, n_rot, q_out=s["q"])
        A.attn_prefill(s["q"], s["cache"], c["start"], c["nh"], out=s["att"], workspace=s["ws"])
        A.o_proj(s["x"], s["att"], s["w"], workspace=s["ows"])
        return s["q"], s["att"], s["x"], s["cache"].k, s["cache"].v
    if kind == "decode":
        return A.attn_decode(s["q"], s["cache"], c["keys"] - 1, c["nh"], out=s["att"], workspace=s["ws"])
    if kind == "batch":
        return A.attn_decode_batch(s["q"], s["batch"], s["lens"], c["nh"], out=s["att"], workspace=s["ws"],
                                   lens_dev=s["lens_dev"])
    if kind == "prefill":
        return A.attn_prefill(s["q"], s["cache"], c["start"], c["nh"], gate=s["gate"], out=s["att"],
                              workspace=s["ws"])
    if kind == "gdn":
        # the gates replace beta in place, as in the engine (another pass takes the sigmoid once more)
        kd, n = c["gh"] * c["gd"], c["gh"]
        G.gdn_gates(s["alpha"], s["beta"], s["dt_bias"], s["ssm_a"], gate=s["gate"])
        rows = G.gdn_conv(s["qkv"], s["line"], s["conv_w"], out=s["rows"], state_out=s["line2"])
        G.gdn_chunk(s["S"], rows[:, :kd], rows[:, kd:2 * kd], rows[:, 2 * kd:], s["gate"], s["beta"], n,
                    out=s["out"], workspace=s["ws"], S_out=s["S2"])
        G.gdn_gated_norm(s["out"], s["z"], s["norm_w"], n, out=s["out"])
        return s["out"], s["S2"], s["line2"]
    if kind == "hybrid":
        for l in s["layers"]:
            G.gdn_decode(l["S"], l["line"], l["line2"], l["qkv"], l["z"], l["alpha"], l["beta"], l["conv_w"],
                         l["dt_bias"], l["ssm_a"], l["norm_w"], c["gh"], y=l["y"], S_out=l["S2"])
        q, k, v = _split(s, c)
        rope, theta, n_rot = _rope_args(c)
        A.attn_decode_rope(q, k, v, s["cache"], c["pos"], c["nh"], rope, theta, n_rot, gate=s["gate"],
                           out=s["att"], workspace=s["ws"])
        return ([(l["y"], l["S2"], l["line2"]) for l in s["layers"]], s["att"], s["cache"].k, s["cache"].v)
    if kind == "rope":
        q, k, v = _split(s, c)
        rope, theta, n_rot = _rope_args(c)
        A.rope_kv_store(s["cache"], q, k, v, c["start"], c["nh"], rope, theta, n_rot, q_out=s["q"])
        return s["q"], s["cache"].k, s["cache"].v
    return A.o_proj(s["x"], s["att"], s["w"])


# ---- what a pass cannot do without ---------------------------------------------------------------

def _causal(T: int, start: int) -> int:
    return T * start + T * (T + 1) // 2


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    if kind == "oproj":
        T, n, k = c["T"], c["hidden"], c["qdim"]
        return {"bytes": 2 * T * k + 2 * n * k + 8 * T * n, "flops": 2 * T * n * k}
    if kind == "gdn" or kind == "hybrid":
        gh, gd = c["gh"], c["gd"]
        conv, state = 3 * gh * gd, gh * gd * gd
        T = c.get("T", 1)
        # qkv, z in, y out, alpha and beta, the state and the delay line before and after; the recurrence's
        # decay, prediction, update and output
        gdn = {"bytes": 4 * (T * (conv + 2 * gh * gd + 2 * gh) + 2 * state + 2 * KW * conv + KW * conv),
               "flops": T * (7 * state + 2 * KW * conv)}
        if kind == "gdn":
            return gdn
    nh, nkv, d = c["nh"], c["nkv"], c["d"]
    qd, kvd = nh * d, nkv * d
    if kind == "hybrid":
        keys = c["pos"] + 1
        return {"bytes": 3 * gdn["bytes"] + 4 * kvd * keys + 4 * (3 * qd + 2 * kvd),
                "flops": 3 * gdn["flops"] + 4 * qd * keys}
    if kind == "token":
        keys = c["pos"] + 1
        return {"bytes": 4 * kvd * keys + 4 * (2 * qd + 2 * kvd) + 2 * qd * qd + 8 * qd,
                "flops": 4 * qd * keys + 2 * qd * qd}
    if kind == "decode":
        return {"bytes": 4 * kvd * c["keys"] + 8 * qd, "flops": 4 * qd * c["keys"]}
    if kind == "batch":
        keys = c["n_seq"] * (c["lo"] + c["hi"]) // 2  # the mean of the drawn lengths
        return {"bytes": 4 * kvd * keys + 8 * qd * c["n_seq"], "flops": 4 * qd * keys}
    T, start = c["T"], c["start"]
    if kind == "rope":
        return {"bytes": T * (qd * (4 + 2) + 2 * kvd * (4 + 2)), "flops": 3 * T * (qd + kvd)}
    if kind == "prefill":
        return {"bytes": 4 * T * qd + 4 * kvd * (start + T) + (4 * T * qd if c["gated"] else 0),
                "flops": 4 * qd * _causal(T, start)}
    # block: the projected rows in, the stored prefix and the new rows, att, W_o once, x in and out
    return {"bytes": 4 * T * (qd + 2 * kvd) + 4 * kvd * (start + T) + 4 * T * qd + 2 * qd * qd + 8 * T * qd,
            "flops": 4 * qd * _causal(T, start) + 2 * T * qd * qd}


def tolerance(case: dict) -> dict:
    # four times what is seen against exact().  Decode and prefill form their products from f16 probabilities
    # (2e-4 of the output), 16-bit outputs add their own rounding (f16 2.1e-4, bf16 1.7e-3), the chunked
    # recurrence's split products leave 2e-5, and o_proj's fp32 sums 2e-7.
    kind = case["kind"]
    if kind == "oproj":
        return {"rel": 1e-6}
    if kind == "gdn":
        return {"rel": 8e-5}
    if kind in ("prefill", "rope"):
        return {"rel": 1e-3 if case["dtype"] == "f16" else 7e-3}
    return {"rel": 8e-4}


# ---- the same in 64 bits -------------------------------------------------------------------------

def _rows_of(cache: A.LayerKV, n: int) -> tuple:
    """The stored keys and values of positions 0..n-1 as float64 [n_kv, n, d]."""
    nkv, stride, d = cache.k.shape
    v = cache.v.view(nkv, stride // 32, d, 32).permute(0, 1, 3, 2).reshape(nkv, stride, d)
    return cache.k[:, :n].double(), v[:, :n].double()


def _rotate(x: torch.Tensor, c: dict, pos: torch.Tensor) -> torch.Tensor:
    """RoPE of float64 rows [T, heads, d] at the positions given; the frequencies are the reference's in float32."""
    d = c["d"]
    span = N_ROT if c["rope"] == "mrope" else d
    f = torch.tensor(c["theta"], dtype=torch.float32).pow(-2.0 * torch.arange(span // 2, dtype=torch.float32) / span)
    ang = (f.cuda()[None, :] * pos.float()[:, None]).double()  # the angle is a float32 product too
    cs, sn = ang.cos()[:, None, :], ang.sin()[:, None, :]
    y = x.clone()
    if c["rope"] == "pairs":
        a, b = x[..., 0::2], x[..., 1::2]
        y[..., 0::2], y[..., 1::2] = a * cs - b * sn, a * sn + b * cs
    else:
        a, b = x[..., :span // 2], x[..., span // 2:span]
        y[..., :span // 2], y[..., span // 2:span] = a * cs - b * sn, a * sn + b * cs
    return y


def _attend(q: torch.Tensor, K: torch.Tensor, V: torch.Tensor, start: int, nh: int) -> torch.Tensor:
    """Causal attention of float64 rows [T, nh * d] at positions start.. over [n_kv, keys, d]."""
    T, d, nkv = q.shape[0], K.shape[2], K.shape[0]
    out = torch.empty_like(q)
    at = torch.arange(K.shape[1], device=q.device)
    for h in range(nh):
        kv = h * nkv // nh
        for t0 in range(0, T, 1024):
            t1 = min(T, t0 + 1024)
            n = start + t1
            p = q[t0:t1, h * d:(h + 1) * d] @ K[kv, :n].t() / math.sqrt(d)
            p.masked_fill_(at[None, :n] > torch.arange(start + t0, n, device=q.device)[:, None], -math.inf)
            out[t0:t1, h * d:(h + 1) * d] = p.softmax(-1) @ V[kv, :n]
    return out


def _store(s: dict, c: dict, k: torch.Tensor, v: torch.Tensor, start: int) -> tuple:
    """The cache after rows k, v (float64 [T, n_kv, d]) are stored at start..: as stored tensors (f16 values) and
    as float64 [n_kv, n, d]."""
    cache, T = s["cache"], k.shape[0]
    kc, vc = cache.k.clone(), cache.v.clone()
    nkv, stride, d = kc.shape
    rows = vc.permute(0, 1, 3, 2).reshape(nkv, stride, d).clone()
    kc[:, start:start + T] = k.permute(1, 0, 2).half()
    rows[:, start:start + T] = v.permute(1, 0, 2).half()
    vc = rows.view(nkv, stride // 32, 32, d).permute(0, 1, 3, 2).contiguous()
    n = start + T
    return kc.double(), vc.double(), kc[:, :n].double(), rows[:, :n].double()


def _rotated(s: dict, c: dict, start: int) -> tuple:
    q, k, v = (t.double().reshape(-1, n, c["d"]) for t, n in zip(_split(s, c), (c["nh"], c["nkv"], c["nkv"])))
    pos = torch.arange(start, start + q.shape[0], device="cuda")
    return _rotate(q, c, pos).reshape(-1, c["nh"] * c["d"]), _rotate(k, c, pos), v


def _gdn_exact(l: dict, gh: int, gd: int) -> tuple:
    """A Gated-DeltaNet layer token by token: (y [T, gh*gd], S after, delay line after)."""
    x = l["qkv"].double().reshape(-1, 3 * gh * gd)
    z = l["z"].double().reshape(-1, gh, gd)
    T = x.shape[0]
    beta = l["beta"].double().reshape(T, gh).sigmoid()
    decay = (torch.log1p((l["alpha"].double().reshape(T, gh) + l["dt_bias"].double()).exp())
             * l["ssm_a"].double()).exp()
    hist = torch.cat([l["line"].double()[1:], x])
    w = l["conv_w"].double()
    conv = sum(hist[i:i + T] * w[:, i] for i in range(KW))
    conv = conv * conv.sigmoid()
    line = torch.cat([l["line"].double(), x])[-KW:]
    q, k, v = conv.reshape(T, 3, gh, gd).unbind(1)
    q = q / q.norm(dim=-1, keepdim=True).clamp_min(G.L2_EPS)
    k = k / k.norm(dim=-1, keepdim=True).clamp_min(G.L2_EPS)
    S, out = l["S"].double(), torch.empty(T, gh, gd, dtype=torch.float64, device="cuda")
    for t in range(T):
        S = S * decay[t][:, None, None]
        delta = (v[t] - (S * k[t][:, None, :]).sum(-1)) * beta[t][:, None]
        S = S + delta[:, :, None] * k[t][:, None, :]
        out[t] = (S * q[t][:, None, :]).sum(-1)
    out = out / math.sqrt(gd)
    y = out * l["norm_w"].double() / (out.square().mean(-1, keepdim=True) + G.L2_EPS).sqrt() * z * z.sigmoid()
    return y.reshape(T, gh * gd), S, line


def exact(case: dict, seed: int):
    c, kind = case, case["kind"]
    s = prepare(case, seed)
    if kind == "oproj":
        return s["x"].double() + s["att"].double() @ s["w"].double().t()
    if kind == "gdn":
        return _gdn_exact(s, c["gh"], c["gd"])
    nh = c["nh"]
    if kind == "token" or kind == "hybrid":
        q, k, v = _rotated(s, c, c["pos"])
        kc, vc, K, V = _store(s, c, k, v, c["pos"])
        att = _attend(q, K, V, c["pos"], nh)[0]
        if kind == "token":
            return att, s["x"].double() + s["w"].double() @ att, kc, vc
        layers = [_gdn_exact(l, c["gh"], c["gd"]) for l in s["layers"]]
        return [(y[0], S, line) for y, S, line in layers], att * s["gate"].double().sigmoid(), kc, vc
    if kind == "block":
        q, k, v = _rotated(s, c, c["start"])
        kc, vc, K, V = _store(s, c, k, v, c["start"])
        att = _attend(q, K, V, c["start"], nh)
        return q, att, s["x"].double() + att @ s["w"].double().t(), kc, vc
    if kind == "rope":
        q, k, v = _rotated(s, c, c["start"])
        kc, vc, _, _ = _store(s, c, k, v, c["start"])
        return q, kc, vc
    if kind == "decode":
        K, V = _rows_of(s["cache"], c["keys"])
        return _attend(s["q"].double()[None], K, V, c["keys"] - 1, nh)[0]
    if kind == "batch":
        out = []
        for i, (n, cache) in enumerate(zip(s["lens"], s["batch"].caches)):
            K, V = _rows_of(cache, n)
            out.append(_attend(s["q"][i].double()[None], K, V, n - 1, nh))
        return torch.cat(out)
    K, V = _rows_of(s["cache"], c["start"] + c["T"])
    att = _attend(s["q"].double(), K, V, c["start"], nh)
    return att * s["gate"].double().sigmoid() if c["gated"] else att
