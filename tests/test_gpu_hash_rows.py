"""The matrix-core hashing kernels (16 rows per wave) and their gradient.

Every slot layout (2 to 6 planes per table, tables that fill a lane group's
slots or leave some empty, one or more sets of tables), row lengths that are
not multiples of 16, row counts around the 16-row groups and the 128-row
workgroups, and few tables of narrow rows, which take the row-per-thread
kernels in one direction or both, against the reference's composition
(src/race_baseline.py:41-44) and its autograd gradient in fp64 on the CPU.
"""
from __future__ import annotations

import math

import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def hash64(x, planes_T, L, K):
    u = torch.tanh(x @ planes_T) / math.sqrt(x.shape[1])
    sign = torch.tensor([[1.0 if (r >> (K - 1 - k)) & 1 else -1.0 for r in range(1 << K)] for k in range(K)],
                        dtype=torch.float64)
    return torch.softmax(u.reshape(len(x), L, K) @ sign, dim=-1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dk, L, K", [(64, 4, 4), (64, 2, 2), (60, 9, 2), (64, 4, 3), (20, 21, 3), (128, 8, 4),
                                      (68, 5, 4), (128, 8, 5), (64, 3, 5), (64, 1, 6), (100, 4, 6), (4, 3, 4),
                                      (32, 1, 4), (36, 1, 4), (16, 2, 3), (20, 4, 2), (12, 1, 3), (16, 1, 3), (28, 1, 5)])
@pytest.mark.parametrize("rows", [1, 17, 128, 333])
def test_rows_and_gradients(race, cuda, dtype, dk, L, K, rows):
    say("hash rows", dtype, dk, L, K, rows)
    gen = torch.Generator().manual_seed(dk + 31 * L + K + rows)
    x = torch.randn(rows, dk, generator=gen).to(dtype)
    planes_T = torch.randn(dk, L * K, generator=gen)
    g = torch.randn(rows, L, 1 << K, generator=gen).to(dtype)
    xd = x.to(cuda).requires_grad_(True)
    probs = race.race_hash_probs(xd, planes_T.to(cuda), L, K)
    (dx,) = torch.autograd.grad(probs, xd, g.to(cuda))

    x64 = x.double().requires_grad_(True)
    want = hash64(x64, planes_T.double(), L, K)
    (want_dx,) = torch.autograd.grad(want, x64, g.double())
    want = want.detach()
    rounding = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    # A projection is a chain of dk / 16 + 2 sums of each lane's products: its
    # error moves u by at most that many roundings of sum |x p| over sqrt(dk),
    # and a probability by 2 per plane and unit of u; the sigmoids and the K
    # products add a few roundings each.
    proj = (x.double().abs() @ planes_T.double().abs()).amax(1) * (dk / 4 + 4) * U  # [rows]
    rel = (2 * K * proj / math.sqrt(dk) + 16 * K * U).reshape(rows, 1, 1)
    err = (probs.double().cpu() - want).abs()
    assert bool((err <= want * (rel + rounding) + 1e-30).all()), err.max()
    # |du_k| <= 2 sum |g p| / sqrt(dk); its factors carry the same errors, and
    # 1 - tanh^2 twice the projection's.
    mass = (g.double().abs() * want).sum(-1)  # [rows, L]
    scale = (mass.repeat_interleave(K, 1) @ planes_T.double().abs().T) * 2 / math.sqrt(dk)  # [rows, dk]
    bound = scale * (2 * rel.reshape(rows, 1) + 4 * proj.reshape(rows, 1) + ((1 << K) + 32) * U)
    err = (dx.double().cpu() - want_dx).abs()
    assert bool((err <= bound + rounding * want_dx.abs() + 1e-30).all()), (err / bound).max()


def test_a_row_only_sees_itself(race, cuda):
    # Infinite and NaN rows next to finite ones in the same 16-row group.
    x = torch.randn(40, 64, device=cuda)
    planes_T = torch.randn(64, 16, device=cuda)
    ref = race.race_hash_probs(x, planes_T, 4, 4)
    y = x.clone()
    y[3] = float("nan")
    y[18, 5] = float("inf")
    got = race.race_hash_probs(y, planes_T, 4, 4)
    keep = torch.ones(40, dtype=torch.bool, device=cuda)
    keep[3] = keep[18] = False
    assert torch.equal(got[keep], ref[keep])
    assert bool(got[3].isnan().all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dk, L, K", [(64, 1, 2), (64, 9, 2), (64, 2, 3), (64, 1, 4), (64, 4, 4), (128, 5, 4),
                                      (64, 2, 5), (60, 3, 6)])
def test_gradient_of_rows_with_infinities(race, cuda, dtype, dk, L, K):
    # A row with one infinity has every plane at tanh(+-inf) = +-1, whose
    # derivative is zero: its gradient is zero, also where the tables leave
    # slots of their set empty, and every other row keeps its bits.
    say("hash rows inf", dtype, dk, L, K)
    gen = torch.Generator().manual_seed(dk + L + K)
    x = torch.randn(40, dk, generator=gen).to(dtype).to(cuda)
    planes_T = torch.randn(dk, L * K, generator=gen).to(cuda)
    g = torch.randn(40, L, 1 << K, generator=gen).to(dtype).to(cuda)
    y = x.clone()
    y[18, 5] = float("inf")
    y[3, dk - 1] = -float("inf")

    def grad(rows):
        rows = rows.requires_grad_(True)
        return torch.autograd.grad(race.race_hash_probs(rows, planes_T, L, K), rows, g)[0]

    ref, got = grad(x), grad(y)
    assert bool((got[[3, 18]] == 0).all()), got[[3, 18]]
    keep = torch.ones(40, dtype=torch.bool, device=cuda)
    keep[[3, 18]] = False
    assert torch.equal(got[keep], ref[keep])
