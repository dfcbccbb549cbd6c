"""The attention work that an inference engine has this library do, as cases that can be
timed and compared: `listed()` names twelve, `draw()` gives others of the same ranges.

Five kinds of call, each through the public entry points:

  decode    ops.DecodeCall / ops.TurboDecodeCall: one new token per sequence over its cache
  prefill   ops.PrefillCall: a prompt, or a chunk that continues a cached one, of one layer
  runstate  runtime.attention_layer_token / prefill_attention_chunk: the drop-in calls with
            host rows over a device cache (one token, or one prefill chunk)
  deltanet  ops.DeltaNetCall: gated DeltaNet over a prompt, or one token of decoding
  encoder   ops.encoder_self_attention: the vision / audio encoders' self-attention

`exact()` evaluates the same inputs in 64 bits with plain torch.
"""
from __future__ import annotations

import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent


def _package():
    name = "gguf_runner_amd"
    if name not in sys.modules:
        d = ROOT / "gguf-runner_amd"
        spec = importlib.util.spec_from_file_location(name, d / "__init__.py", submodule_search_locations=[str(d)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    from gguf_runner_amd import ffi, ops, runtime
    return ffi, ops, runtime


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # The smallest decode: one sequence, 16 / 8 heads, 1024 cached keys, an f32 cache.
        {"name": "decode_f32_1x1024", "kind": "decode", "kv": "f32", "n_seq": 1, "heads": 16, "kv_heads": 8,
         "head_dim": 128, "min_len": 1024, "max_len": 1024, "window": 0},
        # Batched serving over an f16 cache: 16 sequences of ragged lengths up to 32k.
        {"name": "decode_f16_16_ragged_32k", "kind": "decode", "kv": "f16", "n_seq": 16, "heads": 32, "kv_heads": 4,
         "head_dim": 128, "min_len": 1024, "max_len": 32768, "window": 0},
        # The same on the Q8 cache format (one scale per row), a smaller ragged batch of other heads.
        {"name": "decode_q8_7_ragged_16k", "kind": "decode", "kv": "q8", "n_seq": 7, "heads": 32, "kv_heads": 8,
         "head_dim": 128, "min_len": 500, "max_len": 16001, "window": 0},
        # One long conversation on the Turbo format, which is the engine's default.
        {"name": "decode_turbo_2x32k", "kind": "decode", "kv": "turbo", "n_seq": 2, "heads": 32, "kv_heads": 4,
         "head_dim": 128, "min_len": 30011, "max_len": 32768, "window": 0},
        # The longest prompt of the f16 prefill, the largest case.
        {"name": "prefill_f16_8192", "kind": "prefill", "dtype": "f16", "tokens": 8192, "base": 0, "heads": 32,
         "kv_heads": 8, "head_dim": 128, "window": 0, "rope": "adjacent", "norm": False, "bias": False},
        # A sliding-window layer of an 8192-token prompt: bf16, head_dim 256, QK norm.
        {"name": "prefill_bf16_d256_window", "kind": "prefill", "dtype": "bf16", "tokens": 8192, "base": 0, "heads": 8,
         "kv_heads": 4, "head_dim": 256, "window": 1024, "rope": "neox", "norm": True, "bias": False},
        # A follow-up question: a short odd chunk over the rows of the conversation so far,
        # head_dim 64 with the q / k / v biases.
        {"name": "prefill_f16_d64_chunk", "kind": "prefill", "dtype": "f16", "tokens": 203, "base": 3001, "heads": 14,
         "kv_heads": 2, "head_dim": 64, "window": 0, "rope": "neox", "norm": False, "bias": True},
        # The engine's per-token call in its default cache format, host rows in and out.
        {"name": "runstate_token_turbo", "kind": "runstate", "kv": "turbo", "tokens": 1, "base": 1023, "heads": 16,
         "kv_heads": 8, "head_dim": 128},
        # The engine's own prefill chunk (64 tokens) in the middle of a prompt, Q8 cache.
        {"name": "runstate_chunk_q8", "kind": "runstate", "kv": "q8", "tokens": 64, "base": 1984, "heads": 32,
         "kv_heads": 8, "head_dim": 128},
        # DeltaNet over a 4096-token prompt.
        {"name": "deltanet_4096", "kind": "deltanet", "dtype": "bf16", "tokens": 4096, "heads": 16},
        # One token of DeltaNet decoding.
        {"name": "deltanet_step", "kind": "deltanet", "dtype": "bf16", "tokens": 1, "heads": 16},
        # A vision encoder's layer: one image of 4096 patches, 16 heads of 72.
        {"name": "encoder_4096", "kind": "encoder", "n_seq": 1, "tokens": 4096, "heads": 16, "head_dim": 72},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# (query heads, KV heads, head_dim) of the attention layers.
_HEADS = [(16, 8, 128), (32, 8, 128), (32, 4, 128), (14, 2, 64), (8, 4, 256)]


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "runstate", "deltanet", "encoder"])
    if kind == "decode":
        h, g, d = rng.choice(_HEADS)
        kv = rng.choice(["f32", "f16", "bf16", "q8", "q8b", "turbo"])
        n_seq = _log_int(rng, 1, 32)
        top = _log_int(rng, 200, 32768)
        # At most the 276k keys of 4 heads of 128 that the largest listed decode reads.
        top = max(64, min(top, int(275000 * 512 / (g * d) / n_seq)))
        lo = rng.randint(max(1, top // 16), top)
        return {"kind": kind, "kv": kv, "n_seq": n_seq, "heads": h, "kv_heads": g, "head_dim": d, "min_len": lo,
                "max_len": top, "window": 1024 if d == 256 and rng.random() < 0.6 else 0}
    if kind == "prefill":
        h, g, d = rng.choice(_HEADS)
        m = _log_int(rng, 16, 8192)
        base = 0 if rng.random() < 0.5 else _log_int(rng, 1, 8192)
        c = {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "tokens": m, "base": base, "heads": h, "kv_heads": g,
             "head_dim": d, "window": 1024 if d == 256 and rng.random() < 0.6 else 0,
             "rope": "adjacent" if (h, g) == (32, 8) else "neox", "norm": (h, g) in ((16, 8), (32, 4), (8, 4)),
             "bias": d == 64}
        while work(c)["flops"] > 5.4e11:
            c["tokens"] = int(c["tokens"] * 0.7)
        return c
    if kind == "runstate":
        h, g, d = rng.choice(_HEADS)
        m = 1 if rng.random() < 0.5 else _log_int(rng, 2, 512)
        return {"kind": kind, "kv": rng.choice(["f16", "q8", "turbo"]), "tokens": m, "base": _log_int(rng, 30, 4096),
                "heads": h, "kv_heads": g, "head_dim": d}
    if kind == "deltanet":
        h = rng.choice([16, 32])
        t = 1 if rng.random() < 0.3 else _log_int(rng, 2, 65536 // h)
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16", "f32"]), "tokens": t, "heads": h}
    h, d = rng.choice([(16, 72), (16, 64), (12, 64), (16, 80), (8, 128)])
    t = _log_int(rng, 64, 4096)
    n = max(1, min(_log_int(rng, 1, 8), int(4096 * 4096 * 72 * 16 / (t * t * h * max(d, 72)))))
    return {"kind": "encoder", "n_seq": n, "tokens": t, "heads": h, "head_dim": d}


# ---------------------------------------------------------------- sizes

def _lens(case):
    """The batch's cached lengths: uniform in [min_len, max_len], the longest among them."""
    n, lo, hi = case["n_seq"], case["min_len"], case["max_len"]
    rng = np.random.default_rng(1003 + n + hi)
    lens = rng.integers(lo, hi + 1, n)
    lens[int(rng.integers(0, n))] = hi
    w = case["window"]
    return [(max(0, int(x) - w) if w else 0, int(x)) for x in lens]


def _pairs(case):
    m, b, w = case["tokens"], case["base"], case.get("window", 0)
    return sum(min(b + i + 1, w) if w else b + i + 1 for i in range(m))


def _row_bytes(kv, g, d):
    """Bytes of one cached K (or V) row."""
    return {"f32": 4 * g * d, "f16": 2 * g * d, "bf16": 2 * g * d, "q8": g * d + 4, "q8b": g * d + 4 * g * d // 32,
            "turbo": g * (d // 4 + d // 8 + 8)}[kv]


def work(case):
    kind = case["kind"]
    if kind == "deltanet":
        T, H, d = case["tokens"], case["heads"], 128
        el = 4 if case["dtype"] == "f32" else 2
        return {"bytes": T * H * (3 * d * el + 4 * d + 8) + 2 * H * d * d * 4, "flops": 7 * d * d * T * H}
    if kind == "encoder":
        n, T, W = case["n_seq"], case["tokens"], case["heads"] * case["head_dim"]
        return {"bytes": 16 * n * T * W, "flops": 4 * n * T * T * W}
    h, g, d = case["heads"], case["kv_heads"], case["head_dim"]
    if kind == "decode":
        keys = sum(e - s for s, e in _lens(case))
        return {"bytes": 2 * keys * _row_bytes(case["kv"], g, d) + 8 * case["n_seq"] * h * d, "flops": 4 * h * d * keys}
    m, b, w = case["tokens"], case["base"], case.get("window", 0)
    seen = min(b, w) if w else b
    if kind == "prefill":
        n = 2 * m * (h + 2 * g) * d + 4 * m * h * d + 2 * 2 * (m + seen) * g * d
    else:
        n = 4 * m * (h + 2 * g) * d + 4 * m * h * d + 2 * (m + seen) * _row_bytes(case["kv"], g, d)
    return {"bytes": n, "flops": 4 * h * d * _pairs(case)}


# About four times the measured distance of the path from 64 bits: f16 operands (Q and P
# in the prefill, P in the decode over f16 rows) give 2.0e-4 to 2.9e-4; bf16 cache rows
# written by the prefill 1.7e-3 (their own rounding); f32 sums 1e-7 to 3.4e-6; rows
# quantised by the call itself 5.7e-5 (codes whose value lies on a rounding boundary).
def tolerance(case):
    kind, kv = case["kind"], case.get("kv")
    if kind == "prefill":
        return {"rel": 1e-3 if case["dtype"] == "f16" else 2e-3, "max": 0.05}
    if kv == "f16":
        return {"rel": 1e-3, "max": 0.02}
    if kind == "runstate":
        return {"rel": 2e-4, "max": 5e-3}
    return {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------- the cache formats, in plain torch

_M64 = (1 << 64) - 1
_SALTS = (0x9E3779B97F4A7C15, 0xC2B2AE3D27D4EB4F, 0x165667B19E3779F9, 0xD6E8FEB86659FD93)
_CENTROIDS = (-1.510417, -0.45278, 0.45278, 1.510417)
_THRESHOLD = 0.9815985


def _splitmix(x):
    x = (x + 0x9E3779B97F4A7C15) & _M64
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & _M64
    return x ^ (x >> 31)


def _rotations(g, d, dtype, dev):
    """The two rotations of each KV head of layer 0 as matrices [g][d][d] for row vectors
    (x @ R): signs, Walsh-Hadamard transform, signs."""
    sign = np.empty((4, g, d))
    for slot in range(4):
        for j in range(g):
            seed = _splitmix(j ^ _SALTS[slot])
            sign[slot, j] = [1 - 2 * (_splitmix(seed ^ i) & 1) for i in range(d)]
    had = np.ones((1, 1))
    while had.shape[0] < d:
        had = np.block([[had, had], [had, -had]])
    had /= math.sqrt(d)
    rot = [sign[a][:, :, None] * had[None] * sign[a + 1][:, None, :] for a in (0, 2)]
    return [torch.from_numpy(r).to(dev, dtype) for r in rot]


def _turbo_write(x, rot):
    """Rows [..., g, d] -> (codes 0..3, residual sign set, sigma, gamma)."""
    R, P = rot
    y = torch.einsum("...gi,gij->...gj", x, R)
    d = y.shape[-1]
    sigma = (y * y).sum(-1).sqrt() / math.sqrt(d)
    u = y / sigma[..., None]
    code = (u >= -_THRESHOLD).to(torch.uint8) + (u >= 0).to(torch.uint8) + (u >= _THRESHOLD).to(torch.uint8)
    cent = torch.tensor(_CENTROIDS, dtype=torch.float32, device=x.device).to(x.dtype)
    res = y - cent[code.long()] * sigma[..., None]
    gamma = (res * res).sum(-1).sqrt()
    sign = torch.einsum("...gi,gij->...gj", res / gamma[..., None], P) >= 0
    return code, sign, sigma, gamma


def _turbo_read(code, sign, sigma, gamma, rot):
    """The rows that the codes stand for: the attention over them is the one over the codes."""
    R, P = rot
    d = code.shape[-1]
    cent = torch.tensor(_CENTROIDS, dtype=torch.float32, device=code.device).to(sigma.dtype)
    res = (2 * sign.to(sigma.dtype) - 1) * (gamma * math.sqrt(math.pi / 2 / d))[..., None]
    y = cent[code.long()] * sigma[..., None] + torch.einsum("...gj,gij->...gi", res, P)
    return torch.einsum("...gj,gij->...gi", y, R)


def _pack(v, bits):
    n = 8 // bits
    v = v.to(torch.uint8).reshape(*v.shape[:-1], -1, n)
    return sum(v[..., i] << (bits * i) for i in range(n)).to(torch.uint8)


def _unpack(b, bits, d, g):
    n = 8 // bits
    sh = torch.arange(n, device=b.device, dtype=torch.uint8) * bits
    v = (b[..., None] >> sh) & ((1 << bits) - 1)
    return v.reshape(*b.shape[:-1], g, d)


def _q8_write(x, block):
    """Rows [..., g * d] -> (int8 codes, f32 scales), one scale per row or per 32 values."""
    y = x.reshape(*x.shape[:-1], -1, 32) if block else x[..., None, :]
    top = y.abs().amax(-1)
    r = y * (127 / top)[..., None]
    code = (torch.floor(r.abs() + 0.5) * torch.sign(r)).clamp(-127, 127)
    return code.to(torch.int8).reshape(x.shape), top / 127


def _q8_read(code, scale, dtype):
    x = code.to(dtype)
    y = x.reshape(*x.shape[:-1], scale.shape[-1], -1) * scale.to(dtype)[..., None]
    return y.reshape(x.shape)


# ---------------------------------------------------------------- inputs

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _decode_inputs(case, seed):
    dev, gen = torch.device("cuda"), _gen(seed)
    n, h, g, d = case["n_seq"], case["heads"], case["kv_heads"], case["head_dim"]
    lens = _lens(case)
    L = max(e for _, e in lens)
    c = {"q": torch.randn((n, h, d), generator=gen, device=dev)}
    kv = case["kv"]
    for side in "kv":
        if kv in _TORCH:
            c[side] = torch.randn((n, L, g, d), generator=gen, device=dev, dtype=_TORCH[kv])
        elif kv in ("q8", "q8b"):
            x = torch.randn((n, L, g * d), generator=gen, device=dev)
            code, scale = _q8_write(x, kv == "q8b")
            c[side], c[side + "_scale"] = code.view(n, L, g, d), scale.contiguous()
        else:
            rot = _rotations(g, d, torch.float32, dev)
            parts = [_turbo_write(torch.randn((L, g, d), generator=gen, device=dev), rot) for _ in range(n)]
            code, sign, sigma, gamma = (torch.stack(p) for p in zip(*parts))
            c[side] = _pack(code, 2).reshape(n, L, g * d // 4).contiguous()
            c[side + "_sign"] = _pack(sign, 1).reshape(n, L, g * d // 8).contiguous()
            c[side + "_scale"], c[side + "_rnorm"] = sigma.contiguous(), gamma.contiguous()
    c["start"] = torch.tensor([s for s, _ in lens], dtype=torch.int32, device=dev)
    c["end"] = torch.tensor([e for _, e in lens], dtype=torch.int32, device=dev)
    c["max_kv_len"] = max(e - s for s, e in lens)
    return c


def _freqs(theta, d):
    """The engine's f32 frequency table: the f32 power, then the f32 reciprocal."""
    e = (2 * np.arange(d // 2, dtype=np.float32) / np.float32(d)).astype(np.float64)
    return np.float32(1) / np.power(np.float64(np.float32(theta)), e).astype(np.float32)


def _theta(case):
    return {"adjacent": 5e5, "neox": 1e6}[case["rope"]] if not case["window"] else 1e4


def _prefill_inputs(case, seed):
    dev, gen = torch.device("cuda"), _gen(seed)
    m, b, h, g, d = case["tokens"], case["base"], case["heads"], case["kv_heads"], case["head_dim"]
    dt = _TORCH[case["dtype"]]
    rnd = lambda *s, **k: torch.randn(s, generator=gen, device=dev, **k)
    c = {"q": rnd(m, h, d, dtype=dt), "k": rnd(m, g, d, dtype=dt), "v": rnd(m, g, d, dtype=dt),
         "k_cache": rnd(b + m, g, d, dtype=dt), "v_cache": rnd(b + m, g, d, dtype=dt)}
    c["q_norm"], c["k_norm"] = (1 + 0.1 * rnd(d), 1 + 0.1 * rnd(d)) if case["norm"] else (None, None)
    c["q_bias"], c["k_bias"], c["v_bias"] = ((rnd(h * d), rnd(g * d), rnd(g * d)) if case["bias"] else (None, None, None))
    return c


def _runstate_inputs(case, seed):
    """Host rows: the cached tokens' k / v, then the call's q / k / v, and the norm weights."""
    rng = np.random.default_rng(seed)
    m, b, h, g, d = case["tokens"], case["base"], case["heads"], case["kv_heads"], case["head_dim"]
    f = lambda *s: rng.standard_normal(s, dtype=np.float32)
    return {"k_hist": f(b, g * d), "v_hist": f(b, g * d), "q": f(m, h * d), "k": f(m, g * d), "v": f(m, g * d),
            "q_norm": 1 + 0.1 * f(1, d), "k_norm": 1 + 0.1 * f(1, d)}


def _deltanet_inputs(case, seed):
    dev, gen = torch.device("cuda"), _gen(seed)
    T, H, d = case["tokens"], case["heads"], 128
    dt = _TORCH[case["dtype"]]
    rnd = lambda *s, **k: torch.randn(s, generator=gen, device=dev, **k)
    return {"q": rnd(T, H, d, dtype=dt), "k": rnd(T, H, d, dtype=dt), "v": rnd(T, H, d, dtype=dt),
            "gate": -0.1 * torch.rand((T, H), generator=gen, device=dev), "beta": torch.sigmoid(rnd(T, H)),
            "state": 0.1 * rnd(H, d, d)}


def _encoder_inputs(case, seed):
    dev, gen = torch.device("cuda"), _gen(seed)
    n, W = case["n_seq"] * case["tokens"], case["heads"] * case["head_dim"]
    return tuple(torch.randn((n, W), generator=gen, device=dev) for _ in range(3))


def prepare(case, seed):
    ffi, ops, rt = _package()
    dev, kind = torch.device("cuda"), case["kind"]
    if kind == "decode":
        c = _decode_inputs(case, seed)
        out = torch.empty_like(c["q"])
        if case["kv"] == "turbo":
            signs = torch.from_numpy(ops.turbo_sign_table(1, case["kv_heads"], case["head_dim"])).to(dev)
            call = ops.TurboDecodeCall(c["q"], c["k"], c["v"], c["k_sign"], c["v_sign"], c["k_scale"], c["v_scale"],
                                       c["k_rnorm"], c["v_rnorm"], signs, 0, c["start"], c["end"], out,
                                       max_kv_len=c["max_kv_len"])
        else:
            call = ops.DecodeCall(c["q"], c["k"], c["v"], c["start"], c["end"], out, max_kv_len=c["max_kv_len"],
                                  k_scale=c.get("k_scale"), v_scale=c.get("v_scale"), q8_block=case["kv"] == "q8b")
        return {"call": call, "out": out}
    if kind == "prefill":
        c = _prefill_inputs(case, seed)
        d = case["head_dim"]
        out = torch.empty((case["tokens"], case["heads"], d), device=dev)
        freqs = torch.tensor(ops.rope_freqs(_theta(case), d), dtype=torch.float32, device=dev)
        call = ops.PrefillCall(c["q"], c["k"], c["v"], c["k_cache"], c["v_cache"], out, base_pos=case["base"],
                               window=case["window"], rope_dim=d, rope_freqs=freqs,
                               rope_mode=ffi.ROPE_ADJACENT if case["rope"] == "adjacent" else ffi.ROPE_NEOX,
                               q_norm=c["q_norm"], k_norm=c["k_norm"], is_gemma3=d == 256,
                               q_bias=c["q_bias"], k_bias=c["k_bias"], v_bias=c["v_bias"])
        return {"call": call, "out": (out, c["k_cache"], c["v_cache"])}
    if kind == "runstate":
        c = _runstate_inputs(case, seed)
        m, b, d = case["tokens"], case["base"], case["head_dim"]
        p = rt.Config(n_layers=1, n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=d, seq_len=b + m,
                      kv_dtype={"f16": ffi.DTYPE_F16, "q8": ffi.DTYPE_Q8, "turbo": ffi.DTYPE_TURBO}[case["kv"]],
                      rope_mode=ffi.ROPE_NEOX, rope_dim=d, rope_theta=1e6, q_norm=c["q_norm"], k_norm=c["k_norm"])
        s = rt.malloc_run_state(p)
        rt.prefill_attention_chunk(p, s, 0, 0, np.zeros((b, p.q_dim), np.float32), c["k_hist"], c["v_hist"])
        if m == 1:
            s.q[:], s.k[:], s.v[:] = c["q"][0], c["k"][0], c["v"][0]
        return {"p": p, "s": s, "c": c, "base": b, "m": m, "xb": np.zeros((m, p.q_dim), np.float32)}
    if kind == "deltanet":
        c = _deltanet_inputs(case, seed)
        out = torch.empty(c["q"].shape, device=dev)
        call = ops.DeltaNetCall(c["q"], c["k"], c["v"], c["gate"], c["beta"], c["state"], out)
        return {"call": call, "out": (out, c["state"])}
    q, k, v = _encoder_inputs(case, seed)
    out = torch.empty_like(q)
    call = lambda: ops.encoder_self_attention(q, k, v, n_seq=case["n_seq"], tokens=case["tokens"], heads=case["heads"],
                                              head_dim=case["head_dim"], out=out)
    return {"call": call, "out": out}


def run(state):
    if "call" in state:
        state["call"]()
        return state["out"]
    _, _, rt = _package()
    p, s = state["p"], state["s"]
    if state["m"] == 1:
        rt.attention_layer_token(p, s, 0, state["base"])
        return s.xb
    c = state["c"]
    return rt.prefill_attention_chunk(p, s, 0, state["base"], c["q"], c["k"], c["v"], out=state["xb"])


# ---------------------------------------------------------------- the same in 64 bits

def _attend(q, k, v, scale, first, last):
    """q [m][h][d] over k / v [n][g][d] (f64): row i sees keys first[i] .. last[i] - 1."""
    m, h, d = q.shape
    g = k.shape[1]
    out = torch.empty_like(q)
    for j in range(h):
        kj, vj = k[:, j // (h // g)], v[:, j // (h // g)]
        for i in range(0, m, 1024):
            lo, hi = int(first[i:i + 1024].min()), int(last[i:i + 1024].max())
            s = (q[i:i + 1024, j] @ kj[lo:hi].T) * scale
            at = torch.arange(lo, hi, device=q.device)
            seen = (at >= first[i:i + 1024, None]) & (at < last[i:i + 1024, None])
            out[i:i + 1024, j] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ vj[lo:hi]
    return out


def _norm(x, w, eps):
    return x if w is None else x / ((x * x).mean(-1, keepdim=True) + eps).sqrt() * w.double()


def _rope(x, pos, theta, adjacent):
    """x [m][heads][d] rotated at its positions; the frequencies and angles are the path's own f32 values."""
    d = x.shape[-1]
    f = torch.from_numpy(_freqs(theta, d)).to(x.device)
    a = (pos.float()[:, None] * f).double()[:, None]
    c, s = a.cos(), a.sin()
    u, w = (x[..., 0::2], x[..., 1::2]) if adjacent else (x[..., :d // 2], x[..., d // 2:])
    y = (u * c - w * s, u * s + w * c)
    return torch.stack(y, -1).reshape(x.shape) if adjacent else torch.cat(y, -1)


def exact(case, seed):
    dev, kind = torch.device("cuda"), case["kind"]
    if kind == "decode":
        c = _decode_inputs(case, seed)
        n, h, g, d = case["n_seq"], case["heads"], case["kv_heads"], case["head_dim"]
        out = torch.empty((n, h, d), dtype=torch.float64, device=dev)
        rot = _rotations(g, d, torch.float64, dev) if case["kv"] == "turbo" else None
        for i, (s, e) in enumerate(_lens(case)):
            rows = []
            for side in "kv":
                x = c[side][i, s:e]
                if case["kv"] in ("q8", "q8b"):
                    x = _q8_read(x.reshape(e - s, g * d), c[side + "_scale"][i, s:e], torch.float64)
                elif case["kv"] == "turbo":
                    x = _turbo_read(_unpack(x, 2, d, g), _unpack(c[side + "_sign"][i, s:e], 1, d, g),
                                    c[side + "_scale"][i, s:e].double(), c[side + "_rnorm"][i, s:e].double(), rot)
                rows.append(x.double().reshape(e - s, g, d))
            full = torch.tensor([0], device=dev), torch.tensor([e - s], device=dev)
            out[i] = _attend(c["q"][i:i + 1].double(), *rows, 1 / math.sqrt(d), *full)[0]
        return out
    if kind == "prefill":
        c = _prefill_inputs(case, seed)
        m, b, d, w = case["tokens"], case["base"], case["head_dim"], case["window"]
        dt, pos = _TORCH[case["dtype"]], torch.arange(b, b + m, device=dev)
        x = {}
        for n in "qkv":
            x[n] = c[n].double() + (0 if c[n + "_bias"] is None else c[n + "_bias"].double().view(-1, d))
        for n in "qk":
            x[n] = _rope(_norm(x[n], c[n + "_norm"], 1e-6), pos, _theta(case), case["rope"] == "adjacent")
        kc, vc = c["k_cache"].double(), c["v_cache"].double()
        kc[b:], vc[b:] = x["k"], x["v"]
        first = (pos + 1 - w).clamp(min=0) if w else torch.zeros_like(pos)
        out = _attend(x["q"], kc.to(dt).double(), vc.to(dt).double(), 1 / math.sqrt(d), first, pos + 1)
        return out, kc, vc
    if kind == "runstate":
        c = _runstate_inputs(case, seed)
        m, b, h, g, d = case["tokens"], case["base"], case["heads"], case["kv_heads"], case["head_dim"]
        T = lambda a, n: torch.from_numpy(a).to(dev).double().view(-1, n, d)
        qn, kn = (torch.from_numpy(c[n]).to(dev)[0] for n in ("q_norm", "k_norm"))
        pos = torch.arange(b + m, device=dev)
        k = _rope(_norm(T(np.concatenate([c["k_hist"], c["k"]]), g), kn, 1e-6), pos, 1e6, False)
        v = T(np.concatenate([c["v_hist"], c["v"]]), g)
        q = _rope(_norm(T(c["q"], h), qn, 1e-6), pos[b:], 1e6, False)
        kv = []
        for x in (k, v):  # the rows as the cache holds them
            if case["kv"] == "f16":
                x = x.half().double()
            elif case["kv"] == "q8":
                x = _q8_read(*_q8_write(x.reshape(b + m, g * d), False), torch.float64).view(-1, g, d)
            else:
                rot = _rotations(g, d, torch.float64, dev)
                x = _turbo_read(*_turbo_write(x, rot), rot)
            kv.append(x)
        out = _attend(q, *kv, 1 / math.sqrt(d), torch.zeros_like(pos[b:]), pos[b:] + 1)
        out = out.reshape(m, h * d).cpu().numpy()
        return out[0] if m == 1 else out
    if kind == "deltanet":
        c = _deltanet_inputs(case, seed)
        T, H, d = c["q"].shape
        q, k, v = (c[n].double() for n in "qkv")
        q = q / ((q * q).sum(-1, keepdim=True) + 1e-6).sqrt() / math.sqrt(d)
        k = k / ((k * k).sum(-1, keepdim=True) + 1e-6).sqrt()
        decay, beta, S = c["gate"].double().exp(), c["beta"].double(), c["state"].double()
        out = torch.empty((T, H, d), dtype=torch.float64, device=dev)
        for t in range(T):
            S = S * decay[t, :, None, None]
            delta = beta[t, :, None] * (v[t] - (k[t, :, :, None] * S).sum(1))
            S = S + k[t, :, :, None] * delta[:, None, :]
            out[t] = (q[t, :, :, None] * S).sum(1)
        return out, S
    n, T, h, d = case["n_seq"], case["tokens"], case["heads"], case["head_dim"]
    q, k, v = (x.double().view(n, T, h, d) for x in _encoder_inputs(case, seed))
    lo, hi = torch.zeros(T, dtype=torch.int64, device=dev), torch.full((T,), T, device=dev)
    return torch.stack([_attend(q[i], k[i], v[i], 1 / math.sqrt(d), lo, hi) for i in range(n)]).reshape(n * T, h * d)
