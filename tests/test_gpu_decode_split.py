"""Decode steps with a stream's value columns split over two workgroups (wide
values, a separate output state, at most 128 streams) give the in-place step's
bits, whose stream is one workgroup; past 128 streams both are one."""
from __future__ import annotations

import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L, R, d", [(1, 1, 65), (4, 16, 128), (3, 5, 100), (8, 32, 128)])
@pytest.mark.parametrize("N, T", [(1, 1), (7, 9), (128, 3), (129, 2)])
def test_split_step_is_the_whole_step(race, cuda, dtype, L, R, d, N, T):
    say("decode split", dtype, L, R, d, N, T)
    q, k, v = race.make_inputs(N, T, L, R, d, seed=N + T, dtype=dtype, device=cuda)
    gen = torch.Generator(device=cuda).manual_seed(d)
    S = L * R
    state = torch.cat([torch.randn(N, S * d, generator=gen, device=cuda),
                       torch.rand(N, S, generator=gen, device=cuda) + 0.1], dim=1)
    before = state.clone()
    out, new = race.race_fused_fwd_carry(q, k, v, state)
    assert torch.equal(state, before)
    out2, same = race.race_fused_fwd_carry(q, k, v, state, inplace=True)
    assert same is state or same.data_ptr() == state.data_ptr()
    assert torch.equal(out, out2) and torch.equal(new, state)
