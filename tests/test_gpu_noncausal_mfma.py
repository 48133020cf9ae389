"""The non-causal reductions and maps on the fp32 matrix cores.

Widths that fill and that only part-fill the 16-lane vectors, the 16-column
blocks, the 64-column slices and the bf16 operands of eight values (bf16 rows
of 8 m + 4 values are widened to fp32), token counts around the 16- and
32-token steps, and every way the tile records are added (by the maps, by the
separate reduce and finalize), against fp64; the vector-ALU kernels
(kernel="valu") of the same widths under the same bounds.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
EPS = 1e-6


def exact(q, k, v, g):
    """out, dQ, dK, dV in fp64, and for each the sum of its terms' magnitudes."""
    N, T = q.shape[:2]
    q, k = q.reshape(N, T, -1).double(), k.reshape(N, T, -1).double()
    v, g = v.double(), g.double()
    A = k.sum(1) + EPS

    def grads(q, k, v, g, sign):
        E = k.transpose(1, 2) @ v / A[..., None]
        dE = q.transpose(1, 2) @ g
        dB = dE / A[..., None]
        dA = sign * (dE * E).sum(-1) / A
        return (q @ E, g @ E.transpose(1, 2), v @ dB.transpose(1, 2) + dA[:, None], k @ dB)

    return grads(q, k, v, g, -1.0), grads(q, k, v.abs(), g.abs(), 1.0)


def check(got, want, scale, T, S, d, dtype, label):
    # Every value is a sum of products of sums: at most T + S + d roundings of
    # the terms' magnitudes in each of the three nested sums, and a few more
    # from the divisions; bf16 outputs are rounded once.
    rel = 3 * (T + S + d + 16) * U
    for name, a, w, s in zip(("out", "dQ", "dK", "dV"), got, want, scale):
        if a is None:
            continue
        err = (a.reshape(w.shape).double().cpu() - w).abs()
        bound = rel * s + (2.0 ** -8 * w.abs() if dtype == torch.bfloat16 else 0.0) + 1e-30
        assert bool((err <= bound).all()), (label, name, float((err / bound).max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L, R, d", [(1, 4, 4), (3, 4, 20), (2, 8, 64), (3, 16, 96), (5, 20, 36), (4, 16, 64),
                                     (8, 16, 128), (17, 12, 100), (8, 32, 128)])
@pytest.mark.parametrize("N, T", [(2, 1), (3, 33), (2, 130), (2, 1100), (130, 70)])
def test_widths_and_lengths(race, cuda, dtype, L, R, d, N, T):
    say("nc-mfma", dtype, L, R, d, N, T)
    q, k, v, g = race.make_inputs(N, T, L, R, d, seed=N + T + d, dtype=dtype, grad_out=True)
    leaves = [x.to(cuda).requires_grad_(True) for x in (q, k, v)]
    out = race.race_fused_fwd(*leaves, causal=False)
    grads = torch.autograd.grad(out, leaves, g.to(cuda))
    want, scale = exact(q, k, v, g)
    check((out, *grads), want, scale, T, L * R, d, dtype, "mfma")
    valu = race.race_fused_fwd(*(x.detach() for x in leaves), causal=False, kernel="valu")
    check((valu, None, None, None), want, scale, T, L * R, d, dtype, "valu")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tile", [0, 64, 128, 1024])
def test_records_added_by_the_maps_or_before_them(race, cuda, dtype, tile):
    # T = 500: 8 tiles of 64 and 4 of 128 (separate reduce and finalize; the
    # maps), 1 of 1024, and the automatic chunks.
    N, T, L, R, d = 3, 500, 4, 16, 64
    q, k, v, g = race.make_inputs(N, T, L, R, d, seed=5, dtype=dtype, grad_out=True)
    qc, kc, vc, gc = (x.to(cuda) for x in (q, k, v, g))
    out, state = race.race_fused_fwd_with_state(qc, kc, vc, causal=False, tile_tokens=tile)
    want, scale = exact(q, k, v, g)
    full = race.race_noncausal_backward(qc, kc, vc, gc, state, tile_tokens=tile)
    check((out, *full), want, scale, T, L * R, d, dtype, tile)
    B = torch.einsum("nts,ntc->nsc", k.reshape(N, T, -1).double(), v.double()).reshape(N, -1)
    np.testing.assert_allclose(state[:, :-64].double().cpu().numpy(), B.numpy(), atol=T * U * 2 * T)
    for need in ((True, False, False), (False, True, False), (False, False, True), (False, True, True)):
        part = race.race_noncausal_backward(qc, kc, vc, gc, state, need=need, tile_tokens=tile)
        for n, a, b in zip(need, part, full):
            assert torch.equal(a, b) if n else a is None


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L, R, d", [(4, 16, 64), (5, 20, 36), (4, 16, 128), (3, 5, 7)])
@pytest.mark.parametrize("T, tile", [(200, 0), (500, 64), (700, 1024)])
def test_vector_alu_backward(race, cuda, dtype, L, R, d, T, tile):
    # kernel="valu" from the forward to its gradients: the folded passes (4
    # tiles of 64 or one of 1024) and the finalize (8 of 64), each gradient
    # alone, and for widths that have both families other bits than "auto".
    say("nc-valu backward", dtype, L, R, d, T, tile)
    N, S = 2, L * R
    q, k, v, g = race.make_inputs(N, T, L, R, d, seed=T + d, dtype=dtype, grad_out=True)
    leaves = [x.to(cuda).requires_grad_(True) for x in (q, k, v)]
    out = race.race_fused_fwd(*leaves, causal=False, tile_tokens=tile, kernel="valu")
    grads = torch.autograd.grad(out, leaves, g.to(cuda))
    want, scale = exact(q, k, v, g)
    check((out, *grads), want, scale, T, S, d, dtype, "valu")
    qc, kc, vc, gc = (x.to(cuda) for x in (q, k, v, g))
    _, state = race.race_fused_fwd_with_state(qc, kc, vc, causal=False, tile_tokens=tile, kernel="valu")
    for need in ((True, True, True), (True, False, False), (False, True, False), (False, False, True), (False, True, True)):
        part = race.race_noncausal_backward(qc, kc, vc, gc, state, need=need, tile_tokens=tile, kernel="valu")
        for n, a, b in zip(need, part, grads):
            assert torch.equal(a, b) if n else a is None
    auto = race.race_noncausal_backward(qc, kc, vc, gc, state, tile_tokens=tile)
    both = S % 4 == 0 and d % 4 == 0
    assert all(torch.equal(a, b) for a, b in zip(auto, grads)) == (not both)
    with pytest.raises(RuntimeError):
        race.race_noncausal_backward(qc, kc, vc, gc, state, kernel="mfma")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_infinite_values_stay_where_they_are(race, cuda, dtype):
    # An infinity in one value column reaches that column's outputs only, as
    # infinities (the bf16 split of the staged matrix keeps them whole).
    q, k, v = (x.to(cuda) for x in race.make_inputs(2, 100, 4, 16, 64, seed=9, dtype=dtype))
    ref = race.race_fused_fwd(q, k, v, causal=False)
    w = v.clone()
    w[1, 40, 7] = float("inf")
    got = race.race_fused_fwd(q, k, w, causal=False)
    keep = torch.ones_like(ref, dtype=torch.bool)
    keep[1, :, 7] = False
    assert torch.equal(got[keep], ref[keep])
    assert bool((got[1, :, 7] == float("inf")).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L, R, d", [(4, 16, 64), (2, 8, 40), (3, 16, 96), (5, 4, 36), (8, 32, 128)])
def test_infinite_tokens_keep_their_sign(race, cuda, dtype, L, R, d):
    # A token with one infinite value maps to that value's row of the matrix
    # times an infinity: infinities of its signs, no NaN; tokens without one
    # keep their bits.
    say("nc inf tokens", dtype, L, R, d)
    N, T, S = 2, 300, L * R
    q, k, v, g = race.make_inputs(N, T, L, R, d, seed=11, dtype=dtype, grad_out=True)
    q, k = q.reshape(N, T, S), k.reshape(N, T, S)
    qc, kc, vc, gc = (x.to(cuda) for x in (q, k, v, g))
    out, state = race.race_fused_fwd_with_state(qc, kc, vc, causal=False)
    A, B = state[:, S * d:].double().cpu() + EPS, state[:, :S * d].reshape(N, S, d).double().cpu()
    E = B / A[..., None]
    dB = q.double().transpose(1, 2) @ g.double() / A[..., None]
    hit = torch.arange(T) % 3 == 1  # every third token, the infinity in a column of its own

    def spoil(x):
        y, cols = x.clone(), torch.arange(T) % x.shape[-1]
        y[:, hit, cols[hit]] = float("inf") * torch.where(torch.arange(T)[hit] % 2 == 0, 1.0, -1.0).to(y)
        return y

    def check_rows(got, clean, x, m, label):
        # Expected: the sign of the infinity times the matrix row (x's column -> m's row).
        cols = torch.arange(T) % x.shape[-1]
        sign = torch.where(torch.arange(T) % 2 == 0, 1.0, -1.0)
        want = (m[:, cols] * sign[:, None] * float("inf"))[:, hit]
        assert torch.equal(got.double().cpu()[:, hit], want), label
        assert torch.equal(got[:, ~hit], clean[:, ~hit]), label

    # Q in the forward (the sums do not see it).
    check_rows(race.race_fused_fwd(spoil(qc), kc, vc, causal=False), out, q, E, "out")
    clean = race.race_noncausal_backward(qc, kc, vc, gc, state)
    clean = [x.reshape(N, T, -1) for x in clean]
    only = [True, False, False]
    dq = race.race_noncausal_backward(qc, kc, vc, spoil(gc), state, need=only)[0]
    check_rows(dq, clean[0], g, E.transpose(1, 2), "dQ alone")
    dq = race.race_noncausal_backward(qc, kc, vc, spoil(gc), state)[0]
    check_rows(dq, clean[0], g, E.transpose(1, 2), "dQ")
    dk = race.race_noncausal_backward(qc, kc, spoil(vc), gc, state)[1]
    check_rows(dk, clean[1], v, dB.transpose(1, 2), "dK")
    dv = race.race_noncausal_backward(qc, spoil(kc), vc, gc, state)[2]
    check_rows(dv, clean[2], k, dB, "dV")
