"""Short causal sequences at S = d = 64: one launch whose workgroups sum the
tokens before their own tile.

Around the rule's edges (the last tile starting at 512 tokens, six tiles or
512 workgroups, the state from workgroups of its own or from the last tile's),
against fp64: outputs, the prefix records, the state, a
carried state (also advanced in place, which takes the three launches), and
the backward from the saved records against the one that recomputes them.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from gpu_util import FP32_TOL, BF16_TOL, per_stream_rel_err, say, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["auto", "mfma_wg", "mfma_precise"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N, T, tile", [(1, 1, 0), (2, 64, 0), (3, 65, 0), (2, 512, 0), (2, 576, 64), (2, 577, 64),
                                        (2, 641, 128), (1, 1500, 2048), (64, 512, 64), (65, 500, 64), (86, 384, 64),
                                        (300, 64, 0), (520, 33, 0), (130, 300, 0), (257, 600, 512)])
def test_outputs_records_and_states(race, ext, oracle, cuda, kernel, dtype, N, T, tile):
    say("short", kernel, dtype, N, T, tile)
    q, k, v = race.make_inputs(N, T, 4, 16, 64, seed=T + N, dtype=dtype)
    qc, kc, vc = (x.to(cuda) for x in (q, k, v))
    kid = race.ops.KERNELS[kernel]
    out, records, state, used = ext.forward_debug(qc, kc, vc, True, tile, kid)
    ref = oracle.causal_recurrence(to_np(q), to_np(k), to_np(v))
    assert per_stream_rel_err(to_np(out), ref) <= (BF16_TOL if dtype == torch.bfloat16 else FP32_TOL)
    kd, vd = k.reshape(N, T, 64).double(), v.double()
    # fp32 operands as bf16 hi + lo: each within 2^-16 of its value, and the lo
    # * lo product, at most 2^-16, left out; the masses are fp32 sums.
    tol, tol_a = 3 * 2.0 ** -16, (T + 8) * 2.0 ** -24
    for t in range(records.shape[1]):
        n = min(t * used, T)
        B = kd[:, :n].transpose(1, 2) @ vd[:, :n]
        M = kd[:, :n].transpose(1, 2) @ vd[:, :n].abs()
        got = records[:, t, :4096].reshape(N, 64, 64).double().cpu()
        assert bool(((got - B).abs() <= tol * M + 1e-30).all()), t
        A = records[:, t, 4096:4160].double().cpu()
        assert bool(((A - kd[:, :n].sum(1)).abs() <= tol_a * kd[:, :n].sum(1) + 1e-30).all()), t
    B = kd.transpose(1, 2) @ vd
    M = kd.transpose(1, 2) @ vd.abs()
    assert bool(((state[:, :4096].reshape(N, 64, 64).double().cpu() - B).abs() <= tol * M).all())
    assert bool(((state[:, 4096:].double().cpu() - kd.sum(1)).abs() <= tol_a * kd.sum(1)).all())
    # The same without the state, and continued from a state.
    assert torch.equal(ext.forward(qc, kc, vc, True, tile, kid, False)[0], out)
    zero = torch.zeros_like(state)
    out0, state0 = ext.forward_carry(qc, kc, vc, zero, 64 if tile == 0 else tile, 3, False)
    carried = state.clone()
    out1, state1 = ext.forward_carry(qc, kc, vc, carried, 64 if tile == 0 else tile, 3, False)
    out2, state2 = ext.forward_carry(qc, kc, vc, carried, 64 if tile == 0 else tile, 3, True)
    assert torch.allclose(state1, state + state0, rtol=1e-4, atol=1e-4)
    assert torch.allclose(state1, state2, rtol=1e-4, atol=1e-4)
    assert torch.allclose(out1.float(), out2.float(), rtol=2e-2 if dtype == torch.bfloat16 else 1e-3, atol=1e-3)
    twice = oracle.causal_recurrence(*(to_np(torch.cat([x, x], 1)) for x in (q, k, v)))[:, T:]
    assert per_stream_rel_err(to_np(out1), twice) <= (BF16_TOL if dtype == torch.bfloat16 else FP32_TOL)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T, tile", [(500, 64), (576, 64), (577, 64), (600, 512)])
def test_saved_records_and_recomputed_ones_give_the_same_bits(race, ext, cuda, dtype, T, tile):
    q, k, v, g = race.make_inputs(2, T, 4, 16, 64, seed=T, dtype=dtype, device=cuda, grad_out=True)
    _, records, used = ext.forward_with_records(q, k, v, tile, 0)
    saved = ext.causal_backward(q, k, v, g, True, True, True, used, 0, records)
    again = ext.causal_backward(q, k, v, g, True, True, True, used, 0, None)
    assert all(torch.equal(a, b) for a, b in zip(saved, again))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_recomputed_records_of_many_short_streams(race, ext, cuda, dtype):
    # 8 tiles of 64 over more workgroups than CUs: tile sums and a scan, other
    # sums of the same records.
    q, k, v, g = race.make_inputs(40, 512, 4, 16, 64, seed=8, dtype=dtype, device=cuda, grad_out=True)
    _, records, used = ext.forward_with_records(q, k, v, 64, 0)
    saved = ext.causal_backward(q, k, v, g, True, True, True, used, 0, records)
    again = ext.causal_backward(q, k, v, g, True, True, True, used, 0, None)
    for a, b in zip(saved, again):
        assert per_stream_rel_err(to_np(a), to_np(b)) <= (BF16_TOL if dtype == torch.bfloat16 else FP32_TOL)


@pytest.mark.parametrize("T, tile, fwd, bwd", [(512, 64, 1, 4), (576, 64, 1, 4), (577, 64, 3, 5)])
def test_every_launch_is_marked_once(race, cuda, T, tile, fwd, bwd):
    # An event before the first launch and after every one, none for launches
    # that a short sequence does without.
    from race_attention_kernel_amd import abi

    q, k, v, g = race.make_inputs(2, T, 4, 16, 64, seed=T, device=cuda, grad_out=True)
    out, dq, dk, dv = (torch.empty_like(x) for x in (v, q, k, v))
    sh, opts = abi.shape(2, T, 4, 16, 64), abi.options(tile, 0)
    events = [torch.cuda.Event(enable_timing=True) for _ in range(16)]
    stream = torch.cuda.current_stream()
    for e in events:
        e.record(stream)  # creates the handle
    handles = (ctypes.c_void_p * 16)(*(e.cuda_event for e in events))
    status, nbytes, _, _ = abi.fwd_workspace_bytes(sh, True, opts)
    ws = torch.empty(nbytes // 4, device=cuda)
    status, n = abi.fwd_profiled(*(x.data_ptr() for x in (q, k, v, out)), None, sh, True, opts, ws.data_ptr(),
                                 nbytes, stream.cuda_stream, handles)
    assert (status, n) == (0, fwd + 1)
    status, nbytes = abi.causal_bwd_workspace_bytes(sh, opts)
    ws = torch.empty(nbytes // 4, device=cuda)
    status, n = abi.causal_bwd_profiled(*(x.data_ptr() for x in (q, k, v, g, dq, dk, dv)), sh, opts, ws.data_ptr(),
                                        nbytes, stream.cuda_stream, handles)
    assert (status, n) == (0, bwd + 1)
    torch.cuda.synchronize()


@pytest.mark.parametrize("T, tile", [(400, 512), (600, 128), (1100, 512)])
def test_large_calls_give_the_bits_of_small_ones(race, ext, cuda, T, tile):
    # From 201 MB of bf16 tensors on Q and the output go past the caches (one
    # launch of one tile, one of five, three launches): other instructions, the
    # same values.
    N = (3 << 26) // (T * 512) + 1
    say("past the caches", N, T, tile)
    q, k, v = race.make_inputs(N, T, 4, 16, 64, seed=T, dtype=torch.bfloat16, device=cuda)
    big = ext.forward(q, k, v, True, tile, 0, False)[0]
    for n in (0, N - 5):
        small = ext.forward(*(x[n:n + 5].clone() for x in (q, k, v)), True, tile, 0, False)[0]
        assert torch.equal(big[n:n + 5], small)
    assert torch.equal(ext.forward(q, k, v, True, tile, 0, True)[0], big)
