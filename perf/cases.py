"""Performance cases: the calls that a program running a ternary language
model makes, through the package's public entry points.

Kinds (the `kind` of a case):
  linear  one projection: `TernaryLinear.forward` (pack4, pack5, xorsparse) or
          `linear_f32` on weights kept in the compact XorSparse stream (stream)
  mlp     one MLP block: `Mlp.forward`, gate + up, activation, optional
          RMSNorm, requantisation, down
  norm    `FastRmsNorm.forward`
  stack   the projections of a decode step as one planned list: `Stack.run`
  head    the LM head: `Int8Linear.forward` / `Int4Linear.forward`

All of them promise the bits of the CPU path they replace (integer dot
products, two f32 roundings in the epilogue, sums of squares in index order),
so `tolerance` is "exact".  `exact` is the same arithmetic in float64 around
the activation quantiser, whose 8-bit values are part of the result's
definition and follow its f32 scale.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "xor-net_amd"))

import xtern  # noqa: E402
from xtern import (FastRmsNorm, Int4Linear, Int8Linear, Mlp, Stack, TernaryLinear,  # noqa: E402
                   TernaryPackType)

DEV = "cuda:0"
EPS = 1e-5
W_SCALE = 0.8
PACK = {"pack4": TernaryPackType.Pack4, "pack5": TernaryPackType.Pack5}


# --- the cases -------------------------------------------------------------

def listed():
    return [
        # the key / value projection of one decoded token (2560 hidden, 640
        # key-value width): the smallest call of a decode step
        dict(name="kv_token", kind="linear", fmt="pack4", M=1, K=2560, N=640),
        # an 8B-class up projection over a batch of four decoded tokens, the
        # weights kept in the compact XorSparse form to save device memory
        dict(name="xs_stream_batch", kind="linear", fmt="stream", M=4, K=4096, N=14336),
        # a short prompt through a layer whose widths divide nothing
        dict(name="ragged_prompt", kind="linear", fmt="pack5", M=37, K=1003, N=517),
        # the up projection of a 128-token prompt chunk (the prefill shape the
        # benchmark reports)
        dict(name="prompt_chunk", kind="linear", fmt="pack4", M=128, K=2560, N=6912),
        # a 4096-token prompt through an 8B-class XorSparse up projection
        dict(name="long_prompt", kind="linear", fmt="xorsparse", M=4096, K=4096, N=14336),
        # the MLP of one decoded token, ReLU^2 and sub-norm
        dict(name="mlp_token", kind="mlp", fmt="pack4", M=1, K=2560, I=6912, silu=False, norm=True),
        # the same MLP over a 512-token prompt
        dict(name="mlp_prompt", kind="mlp", fmt="pack4", M=512, K=2560, I=6912, silu=False,
             norm=True),
        # a 3B-class MLP with SiLU in the base-3 packing over a 1024-token prompt
        dict(name="mlp_prompt_pack5", kind="mlp", fmt="pack5", M=1024, K=3200, I=8640, silu=True,
             norm=False),
        # the hidden-state norm of a 2048-token prompt
        dict(name="norm_prompt", kind="norm", M=2048, n=2560),
        # one token's 30 layers of projections, each waiting for the one before
        dict(name="decode_chain", kind="stack", fmt="pack4", M=1, layers=30, K=2560, kv=640,
             I=6912, chain=True),
        # eight requests' 30 layers, with the residual stream as the only dependency
        dict(name="decode_batch", kind="stack", fmt="pack4", M=8, layers=30, K=2560, kv=640,
             I=6912, chain=False),
        # logits of eight requests from the Int8 head
        dict(name="head_batch", kind="head", bits=8, M=8, K=2560, N=128256),
    ]


MOST_WORK = 4096 * 4096 * 14336   # M * K * N of the largest listed case


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def width(lo, hi):
        v = log(lo, hi)
        return v if rng.random() < 0.4 else max(64, (v + 32) // 64 * 64)

    kind = rng.choice(["linear"] * 4 + ["mlp"] * 3 + ["norm", "stack", "head"])
    if kind == "linear":
        fmt = rng.choice(["pack4", "pack4", "pack5", "xorsparse", "stream"])
        K, N = width(256, 14336), width(64, 14336)
        M = log(1, 64 if fmt == "stream" else min(4096, max(1, MOST_WORK // (K * N))))
        return dict(kind=kind, fmt=fmt, M=M, K=K, N=N)
    if kind == "mlp":
        return dict(kind=kind, fmt=rng.choice(["pack4", "pack5"]), M=log(1, 2048),
                    K=width(512, 4096), I=width(1024, 10240), silu=rng.random() < 0.5,
                    norm=rng.random() < 0.5)
    if kind == "norm":
        return dict(kind=kind, M=log(1, 4096), n=width(256, 14336))
    if kind == "stack":
        # (in_dims a multiple of 4, as the one-launch plan takes them)
        k = log(32, 80) * 32
        return dict(kind=kind, fmt=rng.choice(["pack4", "pack5"]), M=log(1, 32),
                    layers=log(2, 30), K=k // 20 * 20, kv=k // 4 // 20 * 20,
                    I=int(k * rng.uniform(2.0, 2.7)) // 20 * 20, chain=rng.random() < 0.5)
    return dict(kind=kind, bits=rng.choice([8, 4]), M=log(1, 32), K=width(1024, 2560),
                N=log(8000, 128256))


# --- inputs ----------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _codes(g, N, K):
    """Ternary codes (weight + 1) [N][K], 35 % zeros, as uint8 on the GPU."""
    r = torch.randint(0, 40, (N, K), generator=g, device=DEV, dtype=torch.uint8)
    return (r >= 13).to(torch.uint8) + (r >= 27).to(torch.uint8)


def _rows(g, M, K):
    """Hidden-state rows: normal, with one entry in a hundred 20 times larger."""
    x = torch.randn((M, K), generator=g, device=DEV)
    big = torch.rand((M, K), generator=g, device=DEV) < 0.01
    return torch.where(big, x * 20.0, x)


def _mul_sum(c, f):
    """Sum of digit j of the last axis times 4^j (f = 4) or 3^j (f = 5)."""
    w = torch.tensor([(4 if f == 4 else 3) ** j for j in range(f)], device=DEV, dtype=torch.uint8)
    out = torch.zeros(c.shape[:-1], device=DEV, dtype=torch.uint8)
    for j in range(f):
        out += c[..., j] * w[j]
    return out


def _dense(fmt, g, K, N, keep):
    """A dense TernaryLinear: checkpoint bytes striped over the output rows
    where out_dim allows it, row-packed bytes otherwise.  keep: also the
    weights [N][K] (float64), for `exact`."""
    f = 4 if fmt == "pack4" else 5
    c = _codes(g, N, K)
    if N % f == 0:
        stored = _mul_sum(c.view(f, N // f, K).permute(1, 2, 0), f).cpu().numpy()
        lin = None if keep else TernaryLinear.from_hf_prepacked(stored, K, N, PACK[fmt], W_SCALE,
                                                                False)
    else:
        pad = -K % f
        cp = torch.nn.functional.pad(c, (0, pad), value=0)
        packed = _mul_sum(cp.view(N, -1, f), f).cpu().numpy().ravel()
        lin = None if keep else TernaryLinear.new_direct(packed, K, N, PACK[fmt],
                                                         np.full(N, W_SCALE, np.float32))
    return c.double() - 1.0 if keep else lin


def _sparse(g, K, N, keep):
    """An XorSparse row blob (per row u32 num_blocks, per 64-block u64 mask and
    ceil(nnz / 8) set-order sign bytes), 30 to 70 % zeros per block; keep: the
    weights [N][K] (float64) in its place."""
    nb = (K + 63) // 64
    zero = torch.rand((N, nb, 1), generator=g, device=DEV) * 0.4 + 0.3
    nz = torch.rand((N, nb, 64), generator=g, device=DEV) >= zero
    nz.view(N, nb * 64)[:, K:] = False
    neg = torch.randint(0, 2, (N, nb, 64), generator=g, device=DEV, dtype=torch.uint8)
    nnz = nz.sum(2, keepdim=True)
    neg *= (torch.arange(64, device=DEV) < nnz).to(torch.uint8)   # set order
    if keep:
        rank = (nz.cumsum(2) - 1).clamp_(min=0)
        w = torch.where(nz, 1.0 - 2.0 * torch.gather(neg, 2, rank).double(), 0.0)
        return w.view(N, nb * 64)[:, :K].contiguous()
    bit = torch.tensor([1 << j for j in range(8)], device=DEV, dtype=torch.uint8)

    def bits(v):
        return (v.view(N, nb, 8, 8) * bit).sum(3, dtype=torch.uint8)

    rec = torch.cat([bits(nz.to(torch.uint8)), bits(neg)], 2).view(N, nb * 16)
    there = torch.cat([torch.ones((N, nb, 8), device=DEV, dtype=torch.bool),
                       torch.arange(8, device=DEV) < (nnz + 7) // 8], 2).view(N, nb * 16)
    head = torch.tensor(list(np.uint32(nb).tobytes()), device=DEV, dtype=torch.uint8).expand(N, 4)
    rec = torch.cat([head, rec], 1)
    there = torch.cat([torch.ones((N, 4), device=DEV, dtype=torch.bool), there], 1)
    return rec[there].cpu().numpy()


def _linear(case, g, keep=False):
    K, N = case["K"], case["N"]
    if case["fmt"] in PACK:
        return _dense(case["fmt"], g, K, N, keep)
    blob = _sparse(g, K, N, keep)
    if keep:
        return blob
    ws = np.full(N, W_SCALE, np.float32)
    if case["fmt"] == "stream":
        return xtern.DeviceWeights(xtern.XT_XORSPARSE_STREAM, K, N, blob, ws)
    return TernaryLinear.from_sparse_blob(blob, K, N, ws)


def _head(case, g, keep=False):
    bits, K, N = case["bits"], case["K"], case["N"]
    if bits == 8:
        w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
        raw = w.view(torch.uint8)
    else:
        w = torch.randint(-8, 8, (N, K), generator=g, device=DEV, dtype=torch.int8)
        if K % 2:
            w[:, -1] = 0  # (the last column of an odd in_dim takes no part)
        p = torch.nn.functional.pad(w, (0, K % 2)).view(N, -1, 2) & 15
        raw = (p[..., 0] | (p[..., 1] << 4)).view(torch.uint8)
    sc = torch.rand((N,), generator=g, device=DEV) * 0.002 + 0.001
    if keep:
        return w, sc
    cls = Int8Linear if bits == 8 else Int4Linear
    return cls(raw.cpu().numpy().ravel(), sc.cpu().numpy(), K, N)


def _stack_dims(case):
    K, kv, I = case["K"], case["kv"], case["I"]
    return [("q", K, K), ("k", K, kv), ("v", K, kv), ("o", K, K), ("gate", K, I), ("up", K, I),
            ("down", I, K)]


def _stack(case, g):
    """The projections of `layers` decoder layers.  chain: q/k/v read the
    previous layer's down, o reads q, gate/up read o, down reads gate.
    Otherwise q/k/v and gate/up read the previous layer's down, o and down
    rows that are there before the run (attention and activation outputs)."""
    M, L = case["M"], case["layers"]
    dims = _stack_dims(case)
    w = [{n: _dense(case["fmt"], g, k, m, False).weights for n, k, m in dims} for _ in range(L)]
    y = {n: torch.zeros((L, M, m), device=DEV) for n, _, m in dims}
    x0 = _rows(g, M, case["K"])
    xo = [_rows(g, M, case["K"]) for _ in range(L)]
    xd = [_rows(g, M, case["I"]) for _ in range(L)]
    ops, prev = [], -1
    for l in range(L):
        xin = x0 if prev < 0 else y["down"][l - 1]
        at = len(ops)
        ops.append(([w[l][n] for n in "qkv"], xin, [y[n][l] for n in "qkv"], prev))
        if case["chain"]:
            ops.append(([w[l]["o"]], y["q"][l], [y["o"][l]], at))
            ops.append(([w[l]["gate"], w[l]["up"]], y["o"][l], [y["gate"][l], y["up"][l]], at + 1))
            ops.append(([w[l]["down"]], y["gate"][l], [y["down"][l]], at + 2))
        else:
            ops.append(([w[l]["o"]], xo[l], [y["o"][l]], -1))
            ops.append(([w[l]["gate"], w[l]["up"]], xin, [y["gate"][l], y["up"][l]], prev))
            ops.append(([w[l]["down"]], xd[l], [y["down"][l]], -1))
        prev = at + 3
    return Stack(ops, M), [y[n] for n, _, _ in dims]


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "stack":
        st, ys = _stack(case, g)
        return dict(kind=kind, stack=st, ys=ys)
    if kind == "norm":
        x = _rows(g, case["M"], case["n"])
        return dict(kind=kind, x=x, layer=_norm(g, case["n"]))
    if kind == "mlp":
        K, I = case["K"], case["I"]
        x = _rows(g, case["M"], K)
        gate, up, down = (_dense(case["fmt"], g, a, b, False) for a, b in ((K, I), (K, I), (I, K)))
        layer = Mlp(gate, up, down, _norm(g, I) if case["norm"] else None,
                    "silu" if case["silu"] else "relu2")
        return dict(kind=kind, x=x, layer=layer)
    x = _rows(g, case["M"], case["K"])
    layer = _head(case, g) if kind == "head" else _linear(case, g)
    return dict(kind=kind, x=x, layer=layer, raw=case.get("fmt") == "stream")


def _norm(g, n):
    return FastRmsNorm(torch.rand((n,), generator=g, device=DEV) + 0.5, EPS)


def run(state):
    if state["kind"] == "stack":
        state["stack"].run()
        return state["ys"]
    if state.get("raw"):
        return xtern.linear_f32(state["layer"], state["x"])
    return state["layer"].forward(state["x"])


# --- what a pass cannot do without -----------------------------------------

def _weight_bytes(fmt, K, N):
    if fmt == "pack4":
        return N * ((K + 3) // 4) + 4 * N
    if fmt == "pack5":
        return N * ((K + 4) // 5) + 4 * N
    return N * ((K + 63) // 64) * 12 + 4 * N   # u64 mask + signs of half the lanes, per 64


def work(case):
    kind, M = case["kind"], case["M"]
    if kind == "norm":
        return {"bytes": 8 * M * case["n"] + 4 * case["n"], "flops": 4 * M * case["n"]}
    if kind == "head":
        K, N = case["K"], case["N"]
        return {"bytes": N * K * case["bits"] // 8 + 4 * N + 4 * M * (K + N), "flops": 2 * M * N * K}
    if kind == "linear":
        K, N = case["K"], case["N"]
        return {"bytes": _weight_bytes(case["fmt"], K, N) + 4 * M * (K + N), "flops": 2 * M * N * K}
    K, I = case["K"], case["I"]
    if kind == "mlp":
        return {"bytes": 2 * _weight_bytes(case["fmt"], K, I) + _weight_bytes(case["fmt"], I, K)
                + 8 * M * K, "flops": 6 * M * K * I}
    dims, L = _stack_dims(case), case["layers"]
    byts = sum(_weight_bytes(case["fmt"], k, n) + 4 * M * n for _, k, n in dims)
    return {"bytes": L * byts, "flops": L * sum(2 * M * k * n for _, k, n in dims)}


def tolerance(case):
    return "exact"


# --- the same results in 64 bits -------------------------------------------

def _quant(x):
    """Per-row absmax i8: the f32 scale 127 / max (part of the format), then
    round half to even (the last K % 16 columns half away from zero)."""
    x = x.float()
    mx = x.abs().amax(1, keepdim=True)
    one = torch.ones_like(mx)
    scale = torch.where(mx > 0, 127.0 / mx, one)
    inv = torch.where(mx > 0, mx / 127.0, one).double()
    s = x * scale
    main = x.shape[1] // 16 * 16
    q = torch.round(s)
    q[:, main:] = torch.sign(s[:, main:]) * torch.floor(s[:, main:].abs() + 0.5)
    return q.clamp(-127, 127).double(), inv


def _product(x, w, scale):
    q, inv = _quant(x)
    return (q @ w.T) * inv * scale


def exact(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    ws = float(np.float32(W_SCALE))
    if kind == "norm":
        x = _rows(g, case["M"], case["n"]).double()
        w = _norm(g, case["n"]).weight.double()
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w
    if kind == "stack":
        return None   # (a rounding that differs early on changes 8-bit inputs all the way down)
    if kind == "mlp":
        K, I = case["K"], case["I"]
        x = _rows(g, case["M"], K)
        gate, up, down = (_dense(case["fmt"], g, a, b, True) for a, b in ((K, I), (K, I), (I, K)))
        a, b = _product(x, gate, ws), _product(x, up, ws)
        mid = (a * torch.sigmoid(a) if case["silu"] else torch.relu(a) ** 2) * b
        if case["norm"]:
            mid = mid / torch.sqrt((mid * mid).mean(1, keepdim=True) + EPS) * _norm(g, I).weight.double()
        return _product(mid, down, ws)
    x = _rows(g, case["M"], case["K"])
    if kind == "head":
        w, sc = _head(case, g, keep=True)
        q, inv = _quant(x)
        return torch.cat([(q @ p.double().T) * inv * s.double()
                          for p, s in zip(w.split(16384), sc.split(16384))], 1)
    return _product(x, _linear(case, g, keep=True), ws)
