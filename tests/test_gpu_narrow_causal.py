"""The causal forward on the fp32 matrix cores (up to 64 buckets, widths that
are multiples of 4, no tiled specialization), against fp64.

Widths at the edges of the 16-lane vectors and of the column slices, lengths
around the 16-token steps and the four quarters of a tile, explicit tiles (64
tokens: quarters of one step), a carried state, and infinities, which must not
reach earlier tokens.
"""
from __future__ import annotations

import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
EPS = 1e-6


def causal64(q, k, v, init=None):
    """out [N, T, d] and the sum of its terms' magnitudes, in fp64."""
    N, T = q.shape[:2]
    q, k, v = q.reshape(N, T, -1).double(), k.reshape(N, T, -1).double(), v.double()
    A, B, M = 0.0, 0.0, 0.0
    if init is not None:
        S, d = q.shape[2], v.shape[2]
        B, A = init[:, :S * d].reshape(N, S, d).double(), init[:, S * d:].double()
        M = B.abs()
    outs, mags = [], []
    for t in range(T):
        A = A + k[:, t]
        B = B + k[:, t, :, None] * v[:, t, None]
        M = M + k[:, t, :, None] * v[:, t, None].abs()
        w = (q[:, t] / (A + EPS))[:, None]
        outs.append((w @ B)[:, 0])
        mags.append((w @ M)[:, 0])
    return torch.stack(outs, 1), torch.stack(mags, 1)


def check(out, want, mag, T, S, dtype, label):
    # A value sums S weighted buckets of at most T products, each through a
    # division and a running mass of at most T terms.
    bound = (2 * T + S + 32) * U * mag + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0) + 1e-30
    err = (out.double().cpu() - want).abs()
    assert bool((err <= bound).all()), (label, float((err / bound).max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L, R, d", [(1, 4, 4), (1, 8, 20), (2, 8, 32), (5, 4, 36), (2, 16, 64), (3, 12, 100),
                                     (3, 16, 96), (15, 4, 16), (4, 16, 32), (4, 16, 80)])
@pytest.mark.parametrize("T", [1, 16, 17, 65, 333])
def test_widths_and_lengths(race, cuda, dtype, L, R, d, T):
    say("narrow", dtype, L, R, d, T)
    q, k, v = race.make_inputs(3, T, L, R, d, seed=T + d + L, dtype=dtype)
    want, mag = causal64(q, k, v)
    qc, kc, vc = (x.to(cuda) for x in (q, k, v))
    for tile in (0, 64, 128):
        out, state = race.race_fused_fwd_with_state(qc, kc, vc, True, tile_tokens=tile)
        check(out, want, mag, T, L * R, dtype, tile)
    # Continued from the state of the first half.
    if T > 40:
        h = T // 2
        parts = [x[:, :h].contiguous() for x in (qc, kc, vc)], [x[:, h:].contiguous() for x in (qc, kc, vc)]
        _, st = race.race_fused_fwd_with_state(*parts[0], True)
        out2, st2 = race.race_fused_fwd_carry(*parts[1], st, tile_tokens=64)
        check(out2, want[:, h:], mag[:, h:], T, L * R, dtype, "carry")
        assert torch.allclose(st2, state, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_later_values_do_not_reach_earlier_tokens(race, cuda, dtype, bad):
    # S = 12 leaves four lanes of the bucket vector empty: their products of
    # zero keys with the bad value must not reach the outputs either.
    q, k, v = (x.to(cuda) for x in race.make_inputs(2, 200, 3, 4, 20, seed=3, dtype=dtype))
    ref = race.race_fused_fwd(q, k, v)
    w = v.clone()
    w[0, 71, 5] = bad
    got = race.race_fused_fwd(q, k, w)
    keep = torch.ones_like(ref, dtype=torch.bool)
    keep[0, 71:, 5] = False
    # The step that holds the bad value adds its products one token at a time.
    assert torch.allclose(got[keep].float(), ref[keep].float(), rtol=1e-2 if dtype == torch.bfloat16 else 1e-5,
                          atol=1e-6)
    hit = got[0, 71:, 5]
    assert bool((hit.isnan() if bad != bad else hit == bad).all())


def test_repeats_bit_for_bit(race, cuda):
    q, k, v = (x.to(cuda) for x in race.make_inputs(4, 3000, 2, 8, 32, seed=4))
    ref = race.race_fused_fwd(q, k, v)
    for _ in range(3):
        assert torch.equal(race.race_fused_fwd(q, k, v), ref)
