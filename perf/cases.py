"""The work a user of this package has it do, as timed cases.

Every case goes through the package's public entry points: the causal op, the
non-causal op and their backwards through autograd, the BatchedACE module
(hashing included), Algorithm 1 with the hashing inside, and the decode step.
Sizes are those of the repository's own configurations (inputs.CONFIGS), tests
and benchmark, or generic ones (ragged sequence lengths, narrow heads).

A case is a dict of plain values:
  op      "causal"   race_fused_fwd(..., causal=True), forward only (prefill)
          "bidir"    race_fused_fwd(..., causal=False), forward only
          "module"   BatchedACE.forward (K planes per table, R = 2^K)
          "alg1"     causal_v2.forward (global normalization, K planes)
          "decode"   race_fused_fwd_carry from a carried state
  train   the forward and the gradients w.r.t. every differentiable input
  dtype   "f32" or "bf16"; N streams, T tokens, L tables, R buckets, d columns
  and for the module its causal flag and heads H (N = B * H), for Algorithm 1
  tensor_cores.
"""
from __future__ import annotations

import importlib
import math

import torch

race = importlib.import_module("race-attention-kernel_amd")

EPS = 1e-6
LOGIT_SCALE = 4.0
PREFIX = 1024  # tokens behind a decode step's carried state
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _case(name, op, N, T, L, R, d, dtype, train=False, **more):
    named = {} if name is None else {"name": name}
    return dict(**named, op=op, N=N, T=T, L=L, R=R, d=d, dtype=dtype, train=train, **more)


def listed():
    return [
        # A short prompt: the shortest length of the causal fp32 sweep.
        _case("causal_f32_T512", "causal", 8, 512, 4, 16, 64, "f32"),
        # The headline: the longest length of the causal fp32 sweep.
        _case("causal_f32_T64k", "causal", 8, 65536, 4, 16, 64, "f32"),
        # Long-context prefill of bf16 tokens.
        _case("causal_bf16_T128k", "causal", 8, 131072, 4, 16, 64, "bf16"),
        # Prefill of a small model's narrow heads, a length that is no multiple of anything.
        _case("causal_f32_narrow", "causal", 32, 5001, 2, 8, 32, "f32"),
        # A training step of the causal op, fp32 tokens.
        _case("causal_train_f32", "causal", 8, 16384, 4, 16, 64, "f32", train=True),
        # A training step at language-model scale: many buckets, wide heads, bf16.
        _case("causal_train_bf16_S256", "causal", 128, 16384, 8, 32, 128, "bf16", train=True),
        # A training step of an encoder (classification, vision): batch 32, 12 heads.
        _case("bidir_train_f32", "bidir", 384, 1024, 4, 16, 64, "f32", train=True),
        # The same kind of step on a ragged patch count (24 x 24 patches and a class token), bf16.
        _case("bidir_train_bf16_T577", "bidir", 192, 577, 4, 16, 64, "bf16", train=True),
        # A training step of the causal module, hashing and its gradient included.
        _case("module_causal_train_f32", "module", 8, 16384, 4, 16, 64, "f32", train=True, causal=True, H=8),
        # A training step of the non-causal module: an encoder layer's attention.
        _case("module_bidir_train_f32", "module", 96, 1024, 4, 16, 64, "f32", train=True, causal=False, H=12),
        # Algorithm 1 with the hashing inside, long context, the bf16 feature rounding.
        _case("alg1_bf16_T128k", "alg1", 8, 131072, 4, 16, 64, "bf16", tensor_cores=True),
        # One decode step of every stream of the language-model shape.
        _case("decode_bf16_S256", "decode", 128, 1, 8, 32, 128, "bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges.  Tokens in all (N * T) stay within what
    the listed cases of the kind take, so none costs more than the largest."""
    kind = rng.choice(["causal", "causal", "causal_narrow", "causal_train", "bidir", "bidir_train",
                       "module_causal", "module_bidir", "alg1", "decode"])
    dtype = rng.choice(["f32", "bf16"])
    if kind == "causal":
        L, R = rng.choice([(4, 16), (2, 32), (8, 16), (4, 32), (8, 32)])
        d = rng.choice([64, 64, 128])
        N = _log_int(rng, 1, 128)
        T = _log_int(rng, 64, min(131072, (1 << 20) // N))
        return _case(None, "causal", N, T, L, R, d, dtype)
    if kind == "causal_narrow":
        L, R = rng.choice([(1, 8), (2, 8), (4, 8), (3, 16), (2, 16)])
        d = rng.choice([16, 32, 48, 80, 96])
        N = _log_int(rng, 1, 64)
        T = _log_int(rng, 64, min(16384, (1 << 17) // N))
        return _case(None, "causal", N, T, L, R, d, dtype)
    if kind == "causal_train":
        L, R = rng.choice([(4, 16), (4, 16), (8, 16), (4, 32), (8, 32)])
        d = rng.choice([64, 64, 128])
        N = _log_int(rng, 1, 64)
        T = _log_int(rng, 128, min(65536, (1 << 18) // N))
        return _case(None, "causal", N, T, L, R, d, dtype, train=True)
    if kind in ("bidir", "bidir_train"):
        L, R = rng.choice([(4, 16), (4, 16), (2, 8), (4, 8), (3, 16), (8, 16)])
        d = rng.choice([64, 64, 64, 32, 96, 128])
        N = _log_int(rng, 1, 384)
        T = _log_int(rng, 49, min(16384, (1 << 18) // N))
        return _case(None, "bidir", N, T, L, R, d, dtype, train=kind == "bidir_train")
    if kind in ("module_causal", "module_bidir"):
        L, R = rng.choice([(4, 16), (4, 16), (8, 8), (2, 32), (8, 16)])
        d = rng.choice([64, 64, 128])
        H = rng.choice([1, 4, 8, 12])
        B = _log_int(rng, 1, 16)
        T = _log_int(rng, 64, min(32768, (1 << 17) // (B * H)))
        return _case(None, "module", B * H, T, L, R, d, dtype, train=rng.random() < 0.6,
                     causal=kind == "module_causal", H=H)
    if kind == "alg1":
        K = rng.choice([2, 3, 4, 4, 5])
        N = _log_int(rng, 1, 64)
        T = _log_int(rng, 64, min(131072, (1 << 20) // N))
        return _case(None, "alg1", N, T, rng.choice([1, 2, 4, 4]), 1 << K, rng.choice([64, 64, 128]), "bf16",
                     tensor_cores=rng.random() < 0.5)
    L, R = rng.choice([(4, 16), (8, 16), (8, 32), (2, 8)])
    return _case(None, "decode", _log_int(rng, 1, 512), rng.choice([1, 1, 1, 2, 5, 16]), L, R,
                 rng.choice([64, 64, 128]), dtype)


# ---------------------------------------------------------------------------
# Inputs, from the seed alone.

def _planes(case):
    return int(math.log2(case["R"]))


def _inputs(case, seed):
    """The tensors of a case by name, on the GPU, rounded to its dtype."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    N, T, L, R, d = (case[x] for x in ("N", "T", "L", "R", "d"))
    dt = DTYPES[case["dtype"]]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    def probs(t):
        return torch.softmax(normal(N, t, L, R) * LOGIT_SCALE, dim=-1).to(dt)

    x = {}
    if case["op"] in ("causal", "bidir"):
        x["q"], x["k"], x["v"] = probs(T), probs(T), normal(N, T, d).to(dt)
        if case["train"]:
            x["g"] = normal(N, T, d).to(dt)
    elif case["op"] == "decode":
        pk, pv = probs(PREFIX).float(), normal(N, PREFIX, d)
        pk = pk.reshape(N, PREFIX, L * R)
        B = torch.matmul(pk.transpose(1, 2).contiguous(), pv)
        x["state"] = torch.cat([B.reshape(N, -1), pk.sum(1)], dim=1).contiguous()
        x["q"], x["k"], x["v"] = probs(T), probs(T), normal(N, T, d).to(dt)
    elif case["op"] == "module":
        H = case["H"]
        shape = (1, N // H, T, H, d)
        x["q"], x["k"], x["v"] = (normal(*shape).to(dt) for _ in range(3))
        x["planes"] = normal(L * _planes(case), d)
        if case["train"]:
            x["g"] = normal(*shape).to(dt)
    else:  # alg1
        x["q"], x["k"], x["v"] = (normal(1, N, T, d).to(dt) for _ in range(3))
        x["W"] = normal(L, _planes(case), d) / math.sqrt(d)
        x["beta"] = torch.ones(1, device="cuda")
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    if case["op"] == "module":
        module = race.BatchedACE(case["d"], _planes(case), case["L"], 1, device="cuda", causal=case["causal"])
        module.planes_T.copy_(x["planes"].T)
        x["module"] = module
    if case["train"]:
        for name in ("q", "k", "v"):
            x[name].requires_grad_(True)
    x["case"] = case
    return x


def run(x):
    case = x["case"]
    op = case["op"]
    if op == "decode":
        return race.race_fused_fwd_carry(x["q"], x["k"], x["v"], x["state"])
    if op == "alg1":
        return race.causal_v2.forward(x["q"], x["k"], x["v"], x["W"], x["beta"], 0, case["tensor_cores"])
    if op == "module":
        out = x["module"](x["k"], x["v"], x["q"])
    else:
        out = race.race_fused_fwd(x["q"], x["k"], x["v"], op == "causal")
    if not case["train"]:
        return out
    dq, dk, dv = torch.autograd.grad(out, (x["q"], x["k"], x["v"]), x["g"])
    return out.detach(), dq, dk, dv


# ---------------------------------------------------------------------------

def work(case):
    """Inputs read once, outputs written once; two multiply-adds per bucket and
    column and token (the state and the output) forward, four more backward;
    the module and Algorithm 1 add the projections of the Q and K rows."""
    N, T, L, R, d = (case[x] for x in ("N", "T", "L", "R", "d"))
    es, S, tokens = (4 if case["dtype"] == "f32" else 2), L * R, N * T
    products = 6 if case["train"] else 2
    flops = 2 * tokens * S * d * products
    if case["op"] in ("module", "alg1"):
        rows = 8 if case["train"] else 4  # Q, K, V, out and their gradients
        flops += 2 * tokens * L * _planes(case) * d * (4 if case["train"] else 2)
        return {"bytes": tokens * es * rows * d, "flops": flops}
    if case["op"] == "decode":
        return {"bytes": tokens * es * (2 * S + 2 * d) + 8 * N * (S * d + S), "flops": flops}
    return {"bytes": tokens * es * (2 * S + 2 * d) * (2 if case["train"] else 1), "flops": flops}


def tolerance(case):
    """About four times the largest relative error against exact() measured on
    the listed cases and 96 drawn ones (in brackets)."""
    op, train = case["op"], case["train"]
    if case["dtype"] == "bf16":
        # An output's own rounding alone gives 1.7e-3.
        if op == "module" and train:
            return {"rel": 4e-2}  # gradients through bf16 probabilities [1.0e-2]
        if op in ("bidir", "decode") or (op == "module" and not case["causal"]):
            return {"rel": 7e-3}  # [1.8e-3]
        # Weights and scores rounded to bf16 in the products [2.6e-3]; dK is a
        # sum of terms far larger than itself at the first tokens [8.8e-3].
        return {"rel": 3.5e-2 if train else 1.1e-2}
    if op == "decode" or op == "bidir" or (op == "causal" and (case["L"] * case["R"]) % 64):
        return {"rel": 1.5e-6}  # fp32 products and sums [3.4e-7]
    if op == "module" and not case["causal"]:
        return {"rel": 8e-6 if train else 1.5e-6}  # [2.0e-6, 2.1e-7]
    # Products of bf16 hi + lo pairs, about 2^-17 each [5.0e-6]; dK cancels larger terms [1.7e-5].
    return {"rel": 7e-5 if train else 2e-5}


# ---------------------------------------------------------------------------
# The same functions in 64 bits: plain torch, chunk by chunk.

def _hash64(rows, planes, L, K, beta=None):
    """[..., d] rows -> [..., L * 2^K] corner probabilities (beta: 1 / sqrt(d))."""
    u = torch.tanh(rows @ planes.T) * (1.0 / math.sqrt(rows.shape[-1]) if beta is None else beta)
    sign = torch.tensor([[1.0 if (r >> (K - 1 - p)) & 1 else -1.0 for r in range(1 << K)] for p in range(K)],
                        dtype=rows.dtype, device=rows.device)
    logits = u.reshape(*u.shape[:-1], L, K) @ sign
    return torch.softmax(logits, dim=-1).reshape(*u.shape[:-1], L << K)


def _causal64(q, k, v, init=None, normalize=True, chunk=128, keep=False):
    """out, (A, B) after the last token and, with keep, the state at every chunk
    start.  normalize=False returns (q . B) / (q . A) instead."""
    N, T, S = q.shape
    A = torch.zeros(N, S, dtype=q.dtype, device=q.device)
    B = torch.zeros(N, S, v.shape[2], dtype=q.dtype, device=q.device)
    if init is not None:
        B, A = init[0].clone(), init[1].clone()
    out, states = torch.empty_like(v), []
    for t in range(0, T, chunk):
        qc, kc, vc = q[:, t:t + chunk], k[:, t:t + chunk], v[:, t:t + chunk]
        if keep:
            states.append((A, B))
        Abar = A[:, None] + kc.cumsum(1)
        W = qc / (Abar + EPS) if normalize else qc
        kt = kc.transpose(1, 2).contiguous()
        o = W @ B + torch.tril(W @ kt) @ vc
        if not normalize:
            o = o / (qc * Abar).sum(-1, keepdim=True)
        out[:, t:t + chunk] = o
        A, B = Abar[:, -1], B + kt @ vc
    return out, (A, B), states


def _causal_grads64(q, k, v, g, chunk=128):
    out, (A, B), states = _causal64(q, k, v, chunk=chunk, keep=True)
    Z, Y = torch.zeros_like(B), torch.zeros_like(A)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    for i in range(len(states) - 1, -1, -1):
        c = slice(i * chunk, (i + 1) * chunk)
        qc, kc, vc, gc = q[:, c], k[:, c], v[:, c], g[:, c]
        A, B = states[i]
        r = 1.0 / (A[:, None] + kc.cumsum(1) + EPS)
        W = qc * r
        M = torch.tril(gc @ vc.transpose(1, 2).contiguous())
        P = torch.tril(W @ kc.transpose(1, 2).contiguous())
        dqc = r * (gc @ B.transpose(1, 2).contiguous() + M @ kc)
        alpha = -W * dqc
        suffix = alpha.flip(1).cumsum(1).flip(1)
        dq[:, c] = dqc
        dk[:, c] = vc @ Z.transpose(1, 2).contiguous() + M.transpose(1, 2).contiguous() @ W + suffix + Y[:, None]
        dv[:, c] = kc @ Z + P.transpose(1, 2).contiguous() @ gc
        Z = Z + W.transpose(1, 2).contiguous() @ gc
        Y = Y + alpha.sum(1)
    return out, dq, dk, dv


def _bidir64(q, k, v):
    A, B = k.sum(1), k.transpose(1, 2).contiguous() @ v
    return q @ (B / (A[..., None] + EPS))


def _bidir_grads64(q, k, v, g):
    A, B = k.sum(1) + EPS, k.transpose(1, 2).contiguous() @ v
    E = B / A[..., None]
    dE = q.transpose(1, 2).contiguous() @ g
    dB = dE / A[..., None]
    dA = -(dE * E).sum(-1) / A
    return (q @ E, g @ E.transpose(1, 2).contiguous(), v @ dB.transpose(1, 2).contiguous() + dA[:, None], k @ dB)


def exact(case, seed):
    x = {n: t.double() for n, t in _inputs(case, seed).items()}
    N, T, L, R, d = (case[n] for n in ("N", "T", "L", "R", "d"))
    S, op = L * R, case["op"]
    if op == "decode":
        B, A = x["state"][:, :S * d].reshape(N, S, d), x["state"][:, S * d:]
        out, (A, B), _ = _causal64(x["q"].reshape(N, T, S), x["k"].reshape(N, T, S), x["v"], (B, A))
        return out, torch.cat([B.reshape(N, -1), A], dim=1)
    if op == "alg1":
        planes = x["W"].reshape(L * _planes(case), d)
        q, k = (_hash64(x[n][0], planes, L, _planes(case), float(x["beta"])) for n in ("q", "k"))
        out = _causal64(q, k, x["v"][0], normalize=False)[0]
        return out.reshape(1, N, T, d)
    if op == "module":
        H, K = case["H"], _planes(case)

        def streams(t):  # [1, B, T, H, d] -> [N, T, d]
            return t.permute(0, 1, 3, 2, 4).reshape(N, T, d)

        def back(t):
            return t.reshape(1, N // H, H, T, d).permute(0, 1, 3, 2, 4)

        rows = [streams(x[n]).requires_grad_(case["train"]) for n in ("q", "k")]
        v = streams(x["v"])
        with torch.set_grad_enabled(case["train"]):
            pq, pk = (_hash64(r, x["planes"], L, K) for r in rows)
        q, k = pq.detach(), pk.detach()
        if not case["train"]:
            return back(_causal64(q, k, v)[0] if case["causal"] else _bidir64(q, k, v))
        grads = _causal_grads64 if case["causal"] else _bidir_grads64
        out, dpq, dpk, dv = grads(q, k, v, streams(x["g"]))
        dq, dk = torch.autograd.grad((pq, pk), rows, (dpq, dpk))
        return back(out), back(dq), back(dk), back(dv)
    q, k = x["q"].reshape(N, T, S), x["k"].reshape(N, T, S)
    if not case["train"]:
        return _causal64(q, k, x["v"])[0] if op == "causal" else _bidir64(q, k, x["v"])
    grads = _causal_grads64 if op == "causal" else _bidir_grads64
    out, dq, dk, dv = grads(q, k, x["v"], x["g"])
    return out, dq.reshape(N, T, L, R), dk.reshape(N, T, L, R), dv
