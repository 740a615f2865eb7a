"""The work that this package is used for, as measurable cases.

Each case is a dict of plain values naming one call (or one training step) of
a public entry point at one size.  ``listed`` holds the fixed ones, ``draw``
makes more of the same ranges, ``prepare`` makes the tensors that a program
has in hand before the call, ``run`` makes the call, ``work`` counts the bytes
and operations that the call cannot do without, and ``exact`` gives its result
in 64 bits with plain torch.

Kinds of case:
  norm_fwd    causal normalisation of [B, H, L, L] scores into a given buffer
  norm_train  causal normalisation, forward and backward through autograd
  rowwise     row-wise normalisation of a [rows, cols] matrix
  attn_fwd    fused causal attention, forward only (prefill)
  attn_train  fused causal attention, forward and backward through autograd
  rope        RoPE-fused causal attention, forward only (prefill)
  fp8         fp8 causal attention from 16-bit inputs, quantisation included
  decode      paged single-token attention over the caches
  step        one decode step: append the new token's K and V, then attend
"""
from __future__ import annotations

import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "smooth-attn_amd"))

import smooth_attn as sa  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "fp8": torch.float8_e4m3fn}
PAGE = 16  # cache rows per page
MAX_PAIRS = 4 * 32 * 4096 * 4096  # query-key pairs (before the causal mask) of the largest attention case
EPS = 1e-12


def listed():
    return [
        # The scores of one small layer: the launch and the call count as much as the bytes.
        {"name": "norm_fwd_small", "kind": "norm_fwd", "dtype": "bf16", "B": 2, "H": 8, "L": 512},
        # A training step at a length that is no multiple of anything: rows start at any 2-byte address.
        {"name": "norm_train_odd", "kind": "norm_train", "dtype": "bf16", "B": 2, "H": 16, "L": 1023},
        # The benchmark's training step: forward and backward over 2 GiB of scores.
        {"name": "norm_train_large", "kind": "norm_train", "dtype": "bf16", "B": 4, "H": 16, "L": 4096},
        # Row-wise normalisation of fp32 rows, the only type and shape of the row-wise benchmark.
        {"name": "rowwise_fp32", "kind": "rowwise", "dtype": "fp32", "rows": 65536, "cols": 2048},
        # Prefill of one short prompt with grouped KV heads.
        {"name": "prefill_short", "kind": "attn_fwd", "dtype": "bf16", "B": 1, "Hq": 32, "Hkv": 8, "T": 512, "D": 128,
         "window": 0},
        # A small model's training step: short rows, head dim 64.
        {"name": "train_small_d64", "kind": "attn_train", "dtype": "bf16", "B": 4, "Hq": 12, "Hkv": 12, "T": 1024,
         "D": 64, "window": 0},
        # Fine-tuning with a sliding window and grouped KV heads at a ragged length.
        {"name": "train_window_gqa", "kind": "attn_train", "dtype": "bf16", "B": 2, "Hq": 32, "Hkv": 8, "T": 3000,
         "D": 128, "window": 1024},
        # The benchmark's attention: training at L = 4096, D = 128.
        {"name": "train_large", "kind": "attn_train", "dtype": "bf16", "B": 4, "Hq": 32, "Hkv": 32, "T": 4096,
         "D": 128, "window": 0},
        # Prefill of one long prompt of any length, positions rotated inside.
        {"name": "rope_prefill", "kind": "rope", "dtype": "bf16", "B": 1, "Hq": 32, "Hkv": 8, "T": 8191, "D": 128,
         "window": 0},
        # The fp8 benchmark's sizes, from the bf16 tensors that a caller has.
        {"name": "fp8_prefill", "kind": "fp8", "dtype": "bf16", "B": 2, "Hq": 32, "Hkv": 8, "T": 8192, "D": 128,
         "window": 0},
        # One serving step of a few sequences: launches and host work count.
        {"name": "decode_step_small", "kind": "step", "dtype": "bf16", "cache": "bf16", "B": 8, "Hq": 32, "Hkv": 8,
         "D": 128, "lo": 64, "hi": 2048},
        # The paged benchmark: 64 sequences of 512 to 16384 tokens.
        {"name": "decode_large", "kind": "decode", "dtype": "bf16", "cache": "bf16", "B": 64, "Hq": 32, "Hkv": 8,
         "D": 128, "lo": 512, "hi": 16384},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _length(rng, lo, hi):
    """A row length: as often any number as a multiple of 64."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.5 or n < 64 else n // 64 * 64


def draw(rng):
    kind = rng.choice(["norm_fwd", "norm_train", "rowwise", "attn_fwd", "attn_fwd", "attn_train", "attn_train",
                       "rope", "fp8", "decode", "step"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind in ("norm_fwd", "norm_train"):
        L = _length(rng, 256, 4096)
        BH = max(1, min(256, 64 * 4096 * 4096 // (L * L)))
        H = rng.choice([8, 12, 16])
        return {"kind": kind, "dtype": half, "B": _log_int(rng, 1, max(1, BH // H)), "H": H, "L": L}
    if kind == "rowwise":
        return {"kind": kind, "dtype": "fp32", "rows": _log_int(rng, 512, 65536), "cols": _length(rng, 128, 4096)}
    if kind in ("decode", "step"):
        cache = rng.choice([half, half, "fp8"])
        hi = _log_int(rng, 256, 16384)
        Hq, Hkv = rng.choice([(32, 8), (32, 8), (8, 2), (16, 16)])
        return {"kind": kind, "dtype": "bf16" if cache == "fp8" else half, "cache": cache,
                "B": _log_int(rng, 1, 64), "Hq": Hq, "Hkv": Hkv, "D": rng.choice([64, 128, 128]),
                "lo": max(1, hi // 32), "hi": hi}
    if kind == "fp8":
        half = "bf16"
    D = rng.choice([64, 128, 128]) if kind in ("fp8", "rope") else rng.choice([64, 80, 96, 128, 128])
    T = _length(rng, 256, 8192)
    Hq, Hkv = rng.choice([(32, 8), (32, 32), (16, 2), (12, 12)])
    B = _log_int(rng, 1, max(1, min(16, MAX_PAIRS // (2 * Hq * T * T))))
    window = rng.choice([0, 0, max(32, T // 4)])
    return {"kind": kind, "dtype": half, "B": B, "Hq": Hq, "Hkv": Hkv, "T": T, "D": D, "window": window}


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------
def _randn(gen, shape, dtype, scale=1.0):
    """N(0, scale^2) in dtype (e4m3fn holds the values themselves)."""
    if dtype == torch.float8_e4m3fn:
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16).to(dtype)
    x = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    return x if scale == 1.0 else x.mul_(scale)


def _context_lens(case, gen):
    """Context lengths uniform in [lo, hi], one in each of B equal parts of it,
    in any order: every seed has about the same sum."""
    B, lo, hi = case["B"], case["lo"], case["hi"]
    part = (torch.randperm(B, generator=gen, device="cuda") + torch.rand(B, generator=gen, device="cuda")) / B
    return (lo + part * (hi - lo)).to(torch.int32).clamp_(lo, hi)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    s = {"case": case}
    if kind in ("norm_fwd", "norm_train"):
        shape = (case["B"], case["H"], case["L"], case["L"])
        s["x"] = _randn(gen, shape, dt, 1.0 / math.sqrt(128.0))  # scores of unit-variance q and k times 1/sqrt(D)
        if kind == "norm_fwd":
            s["out"] = torch.empty(shape, device="cuda", dtype=dt)
        else:
            s["x"].requires_grad_(True)
            s["dy"] = _randn(gen, shape, dt)
        return s
    if kind == "rowwise":
        s["x"] = _randn(gen, (case["rows"], case["cols"]), dt)
        s["out"] = torch.empty_like(s["x"])
        return s
    B, Hq, Hkv, D = case["B"], case["Hq"], case["Hkv"], case["D"]
    if kind in ("decode", "step"):
        cdt = DTYPES[case["cache"]]
        lens = _context_lens(case, gen)
        # a pool that holds B sequences of the longest context; the pages of a sequence lie anywhere in it
        width = case["hi"] // PAGE + 1
        total = B * width
        perm = torch.randperm(total, generator=gen, device="cuda").to(torch.int32).view(B, width)
        used = torch.arange(width, device="cuda") <= lens[:, None] // PAGE
        table = torch.where(used, perm, 0)
        s.update(q=_randn(gen, (B, Hq, 1, D), dt), k=_randn(gen, (total, Hkv, PAGE, D), cdt),
                 v=_randn(gen, (total, Hkv, PAGE, D), cdt), table=table, lens=lens)
        if kind == "step":
            s.update(k_new=_randn(gen, (B, Hkv, 1, D), dt), v_new=_randn(gen, (B, Hkv, 1, D), dt))
        return s
    T = case["T"]
    s.update(q=_randn(gen, (B, Hq, T, D), dt), k=_randn(gen, (B, Hkv, T, D), dt), v=_randn(gen, (B, Hkv, T, D), dt))
    if kind == "attn_train":
        for n in "qkv":
            s[n].requires_grad_(True)
        s["do"] = _randn(gen, (B, Hq, T, D), dt)
    if kind == "rope":
        s["cos"], s["sin"] = sa.precompute_rope_cos_sin(D, T)
    return s


# ---------------------------------------------------------------------------
# The calls.
# ---------------------------------------------------------------------------
def _bytes_of(t):
    return t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "norm_fwd":
        return sa.softplus_norm_causal_triton_out(s["out"], s["x"])
    if kind == "norm_train":
        y = sa.softplus_norm_causal(s["x"])
        (dx,) = torch.autograd.grad(y, s["x"], s["dy"])
        return {"y": y.detach(), "dx": dx}
    if kind == "rowwise":
        return sa.softplus_norm_triton_out(s["out"], s["x"])
    if kind == "attn_fwd":
        return sa.sp2norm_flash_attention(s["q"], s["k"], s["v"], window_size=case["window"])
    if kind == "attn_train":
        o = sa.sp2norm_flash_attention(s["q"], s["k"], s["v"], window_size=case["window"])
        dq, dk, dv = torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])
        return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "rope":
        return sa.sp2norm_rope_flash_attention(s["q"], s["k"], s["v"], s["cos"], s["sin"], window_size=case["window"])
    if kind == "fp8":
        return sa.sp2norm_fp8_flash_attention(s["q"], s["k"], s["v"], window_size=case["window"])
    if kind == "decode":
        return sa.sp2norm_paged_attention(s["q"], s["k"], s["v"], s["table"], s["lens"], block_size=PAGE)
    lens = sa.sp2norm_paged_kv_append(s["k"], s["v"], s["k_new"], s["v_new"], s["table"], s["lens"], block_size=PAGE)
    o = sa.sp2norm_paged_attention(s["q"], s["k"], s["v"], s["table"], lens, block_size=PAGE)
    return {"o": o, "lens": lens, "k": _bytes_of(s["k"]), "v": _bytes_of(s["v"])}


# ---------------------------------------------------------------------------
# What a call cannot do without.
# ---------------------------------------------------------------------------
def _pairs(T, window):
    """Query-key pairs of one head under the causal mask and the window."""
    if window <= 0 or window >= T:
        return T * (T + 1) // 2
    return window * (window + 1) // 2 + (T - window) * window


def work(case):
    kind = case["kind"]
    e = 4 if case["dtype"] == "fp32" else 2
    if kind in ("norm_fwd", "norm_train"):
        L = case["L"]
        n, tri = case["B"] * case["H"], L * (L + 1) // 2
        fwd, bwd = e * n * (tri + L * L), e * n * (2 * tri + L * L)  # the causal part in, all of it out
        return {"bytes": fwd + (bwd if kind == "norm_train" else 0), "flops": n * tri * (24 if kind == "norm_train" else 8)}
    if kind == "rowwise":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * e * n, "flops": 8 * n}
    B, Hq, Hkv, D = case["B"], case["Hq"], case["Hkv"], case["D"]
    if kind in ("decode", "step"):
        ce = 1 if case["cache"] == "fp8" else 2
        ctx = B * (case["lo"] + case["hi"]) // 2
        small = B * Hq * D * 4 + B * 4 + (B * Hkv * D * 4 * 2 if kind == "step" else 0)
        return {"bytes": 2 * ce * Hkv * D * ctx + 4 * ctx // PAGE + small, "flops": 4 * Hq * D * ctx}
    T = case["T"]
    qo, kv = B * Hq * T * D * 2, B * Hkv * T * D * 2
    flops = 4 * B * Hq * D * _pairs(T, case["window"])
    if kind == "attn_train":  # forward: q k v in, o out; backward: q k v o do in, dq dk dv out
        return {"bytes": 5 * qo + 6 * kv, "flops": 7 * flops // 2}
    return {"bytes": 2 * qo + 2 * kv, "flops": flops}


def tolerance(case):
    """About four times the distance of a correct result from its 64-bit value."""
    kind = case["kind"]
    if kind == "rowwise":
        return {"rel": 1e-6, "max": 1e-5}  # 32-bit sums and results: 1e-7 measured
    if kind in ("norm_fwd", "norm_train"):
        return {"rel": 6e-3, "max": 0.1}  # 32-bit sums, results in 16 bits: 1.6e-3 in bf16
    # weights and results in 16 bits, sums in 32: 2.3e-3 to 2.8e-3 in bf16, 3.4e-3 where q and k are rotated first
    return {"rel": 1e-2, "max": 0.3}


# ---------------------------------------------------------------------------
# The same results in 64 bits.
# ---------------------------------------------------------------------------
def _norm64(x, causal):
    """Weights over their row sum, its parts as the gradient needs them, alpha = 2, theta = 0.5, power 2."""
    a = 2.0 * (x.double() - 0.5)
    r = torch.sqrt(a * a + 4.0)
    sp = 0.5 * (a + r)
    y = sp * sp
    if causal:
        y = torch.tril(y)
    S = y.sum(-1, keepdim=True) + EPS
    return y / S, sp, r, S


def _norm64_grad(x, dy):
    p, sp, r, S = _norm64(x, True)
    g = dy.double()
    dot = (g * p).sum(-1, keepdim=True)
    return p, torch.tril(4.0 * sp * (sp / r) / S * (g - dot))  # dy/dx = 2 sp * 2 * sp / r


def _rope64(x, cos, sin):
    c, s = cos.double(), sin.double()
    a, b = x.double().chunk(2, dim=-1)
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _fp8_64(x):
    """x as e4m3fn codes with one absmax scale, dequantised.  The two
    divisions are 32-bit ones (64-bit quotients rounded once are the same)."""
    x64 = x.double()
    scale = (x64.abs().amax() / 448.0).float().clamp(min=1e-12).double()
    codes = (x64 / scale).float().clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return codes.double() * scale


def _attn64(q, k, v, do, window):
    """o (and dq, dk, dv where do is given) of one query head, in row parts."""
    T, D = q.shape
    sc = 1.0 / math.sqrt(D)
    o = torch.empty(T, D, dtype=torch.float64, device=q.device)
    grads = [torch.zeros(T, D, dtype=torch.float64, device=q.device) for _ in range(3)] if do is not None else None
    part = 4096
    for r0 in range(0, T, part):
        r1 = min(T, r0 + part)
        c0 = max(0, r0 - window + 1) if window > 0 else 0
        kk, vv = k[c0:r1], v[c0:r1]
        a = sc * (q[r0:r1] @ kk.t().contiguous()) - 0.5
        dist = torch.arange(r0, r1, device=q.device)[:, None] - torch.arange(c0, r1, device=q.device)[None, :]
        keep = (dist >= 0) & (dist < window) if window > 0 else dist >= 0
        r = torch.sqrt(a * a + 1.0)
        y = torch.where(keep, (a + r) ** 2, 0.0)
        R = y.sum(-1, keepdim=True) + EPS
        o[r0:r1] = (y @ vv) / R
        if do is not None:
            g = do[r0:r1]
            p = y / R
            delta = (g * o[r0:r1]).sum(-1, keepdim=True)
            ds = 2.0 * sc * p / r * (g @ vv.t().contiguous() - delta)  # dy/ds = 2 scale y / r
            grads[0][r0:r1] = ds @ kk
            grads[1][c0:r1] += ds.t().contiguous() @ q[r0:r1]
            grads[2][c0:r1] += p.t().contiguous() @ g
    return o, grads


def _paged64(q, k, v, table, lens):
    B, Hq, _, D = q.shape
    Hkv = k.shape[1]
    out = torch.empty(B, Hq, D, dtype=torch.float64, device=q.device)
    for b, n in enumerate(lens.tolist()):
        pages = table[b, : (n + PAGE - 1) // PAGE].long()
        for h in range(Hkv):
            # (16-bit and fp8 values widen exactly)
            kk = k[pages, h].double().reshape(-1, D)[:n]
            vv = v[pages, h].double().reshape(-1, D)[:n]
            G = Hq // Hkv
            a = q[b, h * G:(h + 1) * G, 0].double() @ kk.t().contiguous() / math.sqrt(D) - 0.5
            y = (a + torch.sqrt(a * a + 1.0)) ** 2
            out[b, h * G:(h + 1) * G] = (y @ vv) / (y.sum(-1, keepdim=True) + EPS)
    return out


@torch.no_grad()
def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "rowwise":
        return torch.cat([_norm64(x, False)[0] for x in s["x"].split(8192)])
    if kind in ("norm_fwd", "norm_train"):
        x = s["x"].detach().flatten(0, 1)
        y = torch.empty(x.shape, dtype=torch.float64, device=x.device)
        if kind == "norm_fwd":
            for i in range(x.shape[0]):
                y[i] = _norm64(x[i], True)[0]
            return y.view(s["x"].shape)
        dx = torch.empty_like(y)
        dy = s["dy"].flatten(0, 1)
        for i in range(x.shape[0]):
            y[i], dx[i] = _norm64_grad(x[i], dy[i])
        return {"y": y.view(s["x"].shape), "dx": dx.view(s["x"].shape)}
    if kind in ("decode", "step"):
        if kind == "decode":
            return _paged64(s["q"], s["k"], s["v"], s["table"], s["lens"])
        for b, n in enumerate(s["lens"].tolist()):
            page = int(s["table"][b, n // PAGE])
            for c, new in ((s["k"], s["k_new"]), (s["v"], s["v_new"])):
                _bytes_of(c)[page, :, n % PAGE] = _bytes_of(new[b, :, 0].to(c.dtype))
        o = _paged64(s["q"], s["k"], s["v"], s["table"], s["lens"] + 1)
        return {"o": o, "lens": s["lens"] + 1, "k": _bytes_of(s["k"]), "v": _bytes_of(s["v"])}
    q, k, v = (s[n].detach() for n in "qkv")
    if kind == "rope":
        q, k = _rope64(q, s["cos"], s["sin"]), _rope64(k, s["cos"], s["sin"])
    if kind == "fp8":
        q, k, v = _fp8_64(q), _fp8_64(k), _fp8_64(v)
    B, Hq, T, D = q.shape
    G = Hq // k.shape[1]
    do = s.get("do")
    o = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    grads = [torch.zeros(t.shape, dtype=torch.float64, device=q.device) for t in (q, k, v)] if do is not None else None
    for b in range(B):
        for h in range(Hq):
            kv = h // G
            o[b, h], g = _attn64(q[b, h].double(), k[b, kv].double(), v[b, kv].double(),
                                 None if do is None else do[b, h].double(), case["window"])
            if do is not None:
                grads[0][b, h] = g[0]
                grads[1][b, kv] += g[1]
                grads[2][b, kv] += g[2]
    return o if do is None else {"o": o, "dq": grads[0], "dk": grads[1], "dv": grads[2]}
