"""BatchedACE as one op against the composition of the separate ops, bit for
bit: the copy kernel that lays the heads' rows out as streams (whole 16-byte
rows, rows of a chunk count that is no power of two, batches, ragged run
ends), inputs it does not take (strided, misaligned, one head, one token, odd
row sizes), and which gradients are asked for.
"""
from __future__ import annotations

import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu


def composed(race, ace, K, V, Q):
    """The module's forward out of the package's separate ops."""
    M, B, T, H, d = K.shape

    def rows(x):
        return x.permute(0, 1, 3, 2, 4).contiguous().view(M * B * H, T, d)

    if ace.causal:
        out = race.race_fused_fwd_hashed(rows(K), rows(Q), rows(V), ace.planes_T.t().contiguous(), ace.L)
    else:
        out = race.race_fused_fwd(ace.bucket_probs(rows(Q)), ace.bucket_probs(rows(K)), rows(V), False)
    return out.view(M, B, H, T, d).permute(0, 1, 3, 2, 4)


def compare(race, ace, K, V, Q, need=(True, True, True)):
    ins = [x.detach().requires_grad_(n) for x, n in zip((K, V, Q), need)]
    wanted = [x for x, n in zip(ins, need) if n]
    out, ref = ace(*ins), composed(race, ace, *ins)
    assert out.shape == ref.shape and out.stride() == ref.stride() and torch.equal(out, ref)
    g = torch.randn_like(ref)
    for a, b in zip(torch.autograd.grad(out, wanted, g), torch.autograd.grad(ref, wanted, g)):
        assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("M, B, T, H", [(1, 1, 1, 3), (1, 2, 33, 1), (2, 3, 65, 5), (1, 2, 300, 12)])
def test_module_is_its_parts(race, cuda, dtype, causal, M, B, T, H):
    say("module parts", dtype, causal, M, B, T, H)
    torch.manual_seed(T + H)
    ace = race.BatchedACE(64, 4, 4, M, device=cuda, causal=causal)
    K, V, Q = (torch.randn(M, B, T, H, 64, device=cuda).to(dtype) for _ in range(3))
    compare(race, ace, K, V, Q)


@pytest.mark.parametrize("d, dtype", [(20, torch.float32), (20, torch.bfloat16), (12, torch.float32),
                                      (6, torch.float32), (128, torch.bfloat16)])
def test_row_sizes(race, cuda, d, dtype):
    # 5 chunks a row, 2.5 (through torch), 3, 1.5 (through torch), 16.
    torch.manual_seed(d)
    ace = race.BatchedACE(d, 3, 4, 1, device=cuda, causal=False)
    compare(race, ace, *(torch.randn(1, 2, 77, 3, d, device=cuda).to(dtype) for _ in range(3)))


@pytest.mark.parametrize("causal", [True, False])
def test_inputs_the_copy_kernel_does_not_take(race, cuda, causal):
    torch.manual_seed(1)
    ace = race.BatchedACE(64, 4, 4, 1, device=cuda, causal=causal)
    K, V, Q = (torch.randn(1, 2, 50, 4, 64, device=cuda) for _ in range(3))
    strided = torch.randn(1, 2, 4, 50, 64, device=cuda).transpose(2, 3)
    shifted = torch.randn(1 + K.numel(), device=cuda)[1:].view(K.shape)
    compare(race, ace, strided, V, shifted)
    compare(race, ace, K, V, Q, need=(False, True, False))
    compare(race, ace, K, V, Q, need=(True, False, True))
    with torch.no_grad():
        assert torch.equal(ace(K, V, Q), composed(race, ace, K, V, Q))
    # One head: the permuted rows are the input's own, here misaligned.
    one = torch.randn(1 + 2 * 50 * 64, device=cuda)[1:].view(1, 2, 50, 1, 64)
    out = ace(one, V[:, :, :, :1].contiguous(), one)
    fresh = one.clone()
    assert torch.equal(out, ace(fresh, V[:, :, :, :1].contiguous(), fresh))
    # The inputs may change between the forward and the backward.
    x = [t.clone().requires_grad_(True) for t in (K, V, Q)]
    y = [t * 1.0 for t in x]
    out = ace(*y)
    for t in y:
        t.detach().zero_()
    g = torch.randn_like(out)
    got = torch.autograd.grad(out, x, g)
    want = torch.autograd.grad(ace(*x), x, g)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    with pytest.raises(RuntimeError):
        ace(K, V.to(torch.bfloat16), Q)
    with pytest.raises(RuntimeError):
        ace(K.cpu(), V.cpu(), Q.cpu())


def test_own_bucket_probs_are_used(race, cuda):
    class Uniform(race.BatchedACE):
        def bucket_probs(self, x2):
            return torch.full((*x2.shape[:2], self.L, self.R), 1.0 / self.R, device=x2.device)

    K, V, Q = (torch.randn(1, 1, 40, 2, 64, device=cuda) for _ in range(3))
    ace = Uniform(64, 4, 4, 1, device=cuda, causal=False)
    mean = V.mean(2, keepdim=True).expand_as(V) * ace.L
    assert torch.allclose(ace(K, V, Q), mean, atol=1e-4)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("H", [1, 3])
def test_output_may_be_changed_in_place(race, cuda, causal, H):
    torch.manual_seed(2)
    ace = race.BatchedACE(64, 4, 4, 1, device=cuda, causal=causal)
    x = [torch.randn(1, 2, 40, H, 64, device=cuda).requires_grad_(True) for _ in range(3)]
    out = ace(*x)
    out += x[1]
    out.mul_(2.0)
    got = torch.autograd.grad(out.square().sum(), x)
    ref = (ace(*x) + x[1]) * 2.0
    assert torch.equal(out, ref)
    assert all(torch.equal(a, b) for a, b in zip(got, torch.autograd.grad(ref.square().sum(), x)))


def test_bucket_probs_replaced_on_the_class_are_used(race, cuda, monkeypatch):
    ace = race.BatchedACE(64, 4, 4, 1, device=cuda, causal=False)
    monkeypatch.setattr(race.BatchedACE, "bucket_probs", lambda self, x2: torch.full(
        (*x2.shape[:2], self.L, self.R), 1.0 / self.R, device=x2.device))
    K, V, Q = (torch.randn(1, 1, 40, 2, 64, device=cuda) for _ in range(3))
    mean = V.mean(2, keepdim=True).expand_as(V) * ace.L
    assert torch.allclose(ace(K, V, Q), mean, atol=1e-4)


def saved_floats(fn):
    """Elements a call saves for its backward, each storage once."""
    seen = {}

    def pack(t):
        seen[t.untyped_storage().data_ptr()] = t.untyped_storage().nbytes() // 4
        return t

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        out = fn()
    return sum(seen.values()), out


@pytest.mark.parametrize("need", [(True, False, False), (False, True, False), (False, False, True)])
def test_rows_that_no_gradient_reads_are_not_saved(race, cuda, need):
    # The separate ops keep the rows of a hashing only for its own gradient.
    torch.manual_seed(3)
    ace = race.BatchedACE(64, 4, 4, 1, device=cuda, causal=False)
    x = [torch.randn(1, 2, 40, 3, 64, device=cuda).requires_grad_(n) for n in need]
    got, _ = saved_floats(lambda: ace(*x))
    ref, _ = saved_floats(lambda: composed(race, ace, *x))
    assert got <= ref, (got, ref)
    compare(race, ace, *x, need=need)


@pytest.mark.parametrize("causal", [True, False])
def test_no_grad_keeps_nothing(race, ext, cuda, causal, monkeypatch):
    # Inputs that require a gradient, in a forward without one: no state or
    # records are asked for.
    ace = race.BatchedACE(64, 4, 4, 1, device=cuda, causal=causal)
    x = [torch.randn(1, 1, 40, 2, 64, device=cuda).requires_grad_(True) for _ in range(3)]
    kept = []

    class Spy:
        def __getattr__(self, name):
            f = getattr(ext, name)
            if name != "module_forward":
                return f

            def call(*a):
                r = f(*a)
                kept.append(len(r[1]))
                return r

            return call

    monkeypatch.setattr(race.ops._lib, "ext", lambda: Spy())
    with torch.no_grad():
        out = ace(*x)
    assert kept == [0] and not out.requires_grad
    ace(*x)
    assert kept[1] > 0
