"""CPU emulation of the index math of the row passes on the matrix cores (no
GPU): noncausal_mfma.hip, hash_rows.hip, narrow_causal.hip and pack_heads.hip.

Each mapping is restated from the function named in its test and carried
through a model of the instructions it feeds: the products must come out as
plain matrix products, the turns through LDS must return every value once and
spread over the banks, and a planted mistake must fail.

The instruction model: a lane is (g, lr) = (lane / 16, lane % 16); a 16x16
matrix instruction takes A[row lr][k of g] and B[k of g][column lr] from each
lane and returns D[4 g + r][lr], with one k per lane group in fp32 (4 in all)
and eight in bf16 (32 in all).
"""
from __future__ import annotations

from collections import Counter

import numpy as np
import pytest

LANES = [(lane, lane >> 4, lane & 15) for lane in range(64)]


def mfma(a, b, acc):
    """acc[lane][r] += the product of a[lane][k], b[lane][k] (k values per lane group)."""
    A = np.zeros((16, 4, len(a[0])))
    B = np.zeros((4, len(a[0]), 16))
    for lane, g, lr in LANES:
        A[lr, g] = a[lane]
        B[g, :, lr] = b[lane]
    D = np.einsum("mgk,gkn->mn", A, B)
    for lane, g, lr in LANES:
        acc[lane] += D[4 * g:4 * g + 4, lr]
    return acc


def zeros():
    return np.zeros((64, 4))


def worst_bank_use(slots, unit):
    """Most accesses to one bank by the 16 lanes served together, for units of
    `unit` bytes at slot numbers `slots` (64 banks of 4 bytes)."""
    worst = 0
    for i in range(0, 64, 16):
        use = Counter()
        for s in set(slots[i:i + 16]):
            for w in range(unit // 4):
                use[(s * unit // 4 + w) % 64] += 1
        worst = max(worst, max(use.values()))
    return worst


# ---------------------------------------------------------------------------
# noncausal_mfma.hip


@pytest.mark.parametrize("N, per", [(1, 1), (1, 7), (8, 3), (9, 2), (13, 5), (384, 2), (192, 1)])
def test_stream_block_takes_every_block_once(N, per):
    seen, xcd = set(), {}
    for wg in range(N * per):
        group = wg // (8 * per)
        inside = wg - group * 8 * per
        streams = min(8, N - 8 * group)
        n, blk = 8 * group + inside % streams, inside // streams
        seen.add((n, blk))
        if streams == 8:
            xcd.setdefault(n, set()).add(wg % 8)
    assert seen == {(n, b) for n in range(N) for b in range(per)}
    assert all(len(x) == 1 for x in xcd.values())  # a stream's blocks share an XCD


def map_rows(NJ, b16, es):
    per = 8 if b16 else 4
    ops = (NJ + 1) // 2 if b16 else NJ
    return per, ops, 4 * ops, per * es


@pytest.mark.parametrize("NJ", [1, 2, 4, 8])
@pytest.mark.parametrize("b16, es", [(False, 4), (False, 2), (True, 2)])
def test_turn_gives_each_lane_its_operands(NJ, b16, es):
    # MapRows::load, at, turn: 16 rows of units loaded whole, read by token.
    per, ops, units, unit = map_rows(NJ, b16, es)

    def at(row, u, swizzle=True):
        return row * units + (u ^ (row & (units - 1)) if swizzle else u)

    lds = {}
    for i in range(ops):
        slots = []
        for lane, _, _ in LANES:
            u = i * 64 + lane
            slots.append(at(u // units, u % units))
            assert slots[-1] not in lds
            lds[slots[-1]] = (u // units, u % units)
        assert worst_bank_use(slots, unit) <= 2
    assert len(lds) == 16 * units
    for j in range(ops):
        slots = [at(lr, 4 * j + g) for _, g, lr in LANES]
        assert [lds[s] for s in slots] == [(lr, 4 * j + g) for _, g, lr in LANES]
        # 16 rows of a few units are shorter than the banks: no worse than the
        # rows' own overlap.
        assert worst_bank_use(slots, unit) <= max(2, 16 // units)
    if units >= 8:
        plain = [at(lr, g, swizzle=False) for _, g, lr in LANES]
        assert worst_bank_use(plain, unit) > 2  # without the swizzle they collide


def put_matrix(M, NCB, b16, across):
    """The staged matrix, flat, of M [k][c] as put_matrix lays it out (bf16:
    [term] kept as a trailing axis of (term, k, c) tags)."""
    K, C = M
    dst = {}
    step = range(0, C, 4) if across else range(C)
    for k in (range(K) if across else range(0, K, 4)):
        for c in step:
            cb, lr = c >> 4, c & 15
            if b16:
                j, g, e = k >> 5, (k >> 3) & 3, k & 7
                for s in range(3):
                    at = (((j * NCB + cb) * 3 + s) * 64 + 16 * g + lr) * 8 + e
                    for i in range(4):
                        key, val = (at + 8 * i, (s, k, c + i)) if across else (at + i, (s, k + i, c))
                        assert key not in dst
                        dst[key] = val
            else:
                j, g, e = k >> 4, (k >> 2) & 3, k & 3
                for i in range(4):
                    if across:
                        key, val = ((j * NCB + cb) * 64 + 16 * g + lr + i) * 4 + e, (0, k, c + i)
                    else:
                        key, val = ((j * NCB + cb) * 64 + 16 * g + lr) * 4 + i, (0, k + i, c)
                    assert key not in dst
                    dst[key] = val
    return dst


@pytest.mark.parametrize("NJ, NCB", [(1, 1), (2, 4), (4, 2), (4, 4)])
@pytest.mark.parametrize("b16", [False, True])
def test_staged_matrix_times_rows_is_the_product(NJ, NCB, b16):
    per, ops, _, _ = map_rows(NJ, b16, 2 if b16 else 4)
    K, C = (32 * ops if b16 else 16 * NJ), 16 * NCB
    flat = put_matrix((K, C), NCB, b16, across=True)
    assert flat == put_matrix((K, C), NCB, b16, across=False)
    assert sorted(flat) == list(range(K * C * (3 if b16 else 1)))
    rng = np.random.default_rng(NJ + NCB)
    terms = rng.standard_normal((3 if b16 else 1, K, C))
    X = rng.standard_normal((16, K))

    def m(entry, e):
        return terms[flat[entry * per + e]]

    acc = [zeros() for _ in range(NCB)]
    whole = [zeros() for _ in range(NCB)]
    for j in range(ops):
        x = [X[lr, 4 * per * j + per * g:4 * per * j + per * g + per] for _, g, lr in LANES]
        for cb in range(NCB):
            if b16:
                for s in range(3):  # MapRows::times
                    a = [[m(((j * NCB + cb) * 3 + s) * 64 + lane, e) for e in range(8)] for lane, _, _ in LANES]
                    mfma(a, x, acc[cb])
            else:
                for e in range(4):
                    a = [[m((j * NCB + cb) * 64 + lane, e)] for lane, _, _ in LANES]
                    mfma(a, [[v[e]] for v in x], acc[cb])
    if b16:  # whole_products: half operands, the terms put together
        for cb in range(NCB):
            for h in range(2 * ops):
                j = h >> 1
                for e in range(4):
                    a = [[sum(m(((j * NCB + cb) * 3 + s) * 64 + lane, 4 * (h & 1) + e) for s in range(3))]
                         for lane, _, _ in LANES]
                    b = [[X[lr, 32 * j + 8 * g + 4 * (h & 1) + e]] for _, g, lr in LANES]
                    mfma(a, b, whole[cb])
    want = X @ terms.sum(0)
    for result in (acc, whole) if b16 else (acc,):
        for cb in range(NCB):
            for lane, g, lr in LANES:
                np.testing.assert_allclose(result[cb][lane], want[lr, 16 * cb + 4 * g:16 * cb + 4 * g + 4], atol=1e-10)


@pytest.mark.parametrize("NCB", [1, 2, 4])
def test_result_rows_leave_whole(NCB):
    # OutRows: results of (token lr, unit 4 cb + g) through LDS to whole rows.
    units = 4 * NCB

    def at(row, u):
        return row * units + (u ^ (row & (units - 1)))

    lds = {at(lr, 4 * cb + g): (lr, 4 * cb + g) for cb in range(NCB) for _, g, lr in LANES}
    assert len(lds) == 16 * units
    out = [lds[at((i * 64 + lane) // units, (i * 64 + lane) % units)] for i in range(NCB) for lane in range(64)]
    assert out == [(r, u) for r in range(16) for u in range(units)]


def test_query_side_turns_the_reductions_rows_into_map_operands():
    # nc_query64_kernel: rows 4 i + g, columns 4 lr .. stored by unit, read as
    # MapRows operands (one unit in fp32, two in bf16).
    for tokens, per_op, map_units in ((16, 1, 16), (32, 2, 8)):
        def at(row, u):
            return row * 16 + per_op * ((u // per_op) ^ (row & (map_units - 1))) + u % per_op

        lds = {at(4 * i + g, lr): (4 * i + g, lr) for i in range(tokens // 4) for _, g, lr in LANES}
        assert len(lds) == 16 * tokens
        for h in range(tokens // 16):
            for j in range(4 // per_op):
                for _, g, lr in LANES:
                    first = at(16 * h + lr, per_op * (4 * j + g))
                    got = [lds[first + p] for p in range(per_op)]
                    assert got == [(16 * h + lr, per_op * (4 * j + g) + p) for p in range(per_op)]


@pytest.mark.parametrize("EA, EB", [(2, 2), (2, 4), (4, 2), (4, 4)])
@pytest.mark.parametrize("b16", [False, True])
def test_reduction_blocks_are_the_outer_sums(EA, EB, b16):
    # Columns, Outer::add and spill: lane (g, lr) loads tokens 4 i + g, columns
    # EA lr .. and EB lr ..; block (a, b) holds rows EA m + a, columns EB n + b.
    tokens = 32 if b16 else 16
    rng = np.random.default_rng(EA + EB)
    x, y = rng.standard_normal((tokens, 16 * EA)), rng.standard_normal((tokens, 16 * EB))
    R = np.full((16 * EA, 16 * EB), np.nan)
    for a in range(EA):
        for b in range(EB):
            acc = zeros()
            xs = [[x[4 * i + g, EA * lr + a] for i in range(tokens // 4)] for _, g, lr in LANES]
            ys = [[y[4 * i + g, EB * lr + b] for i in range(tokens // 4)] for _, g, lr in LANES]
            if b16:
                mfma(xs, ys, acc)
            else:
                for i in range(4):
                    mfma([[v[i]] for v in xs], [[v[i]] for v in ys], acc)
            for lane, g, lr in LANES:
                for r in range(4):
                    R[EA * (4 * g + r) + a, EB * lr + b] = acc[lane][r]
    np.testing.assert_allclose(R, x.T @ y, atol=1e-10)


def test_three_terms_are_the_value():
    # split3: truncated bf16 terms; exact from 2^-110 up, infinities in one term.
    def top(v):
        return (np.float32(v).view(np.uint32) & np.uint32(0xffff0000)).view(np.float32)

    rng = np.random.default_rng(3)
    x = (rng.standard_normal(20000) * 2.0 ** rng.integers(-100, 100, 20000)).astype(np.float32)
    hi = np.array([top(v) for v in x])
    r1 = x - hi
    mid = np.array([top(v) for v in r1])
    lo = np.array([top(v) for v in r1 - mid])
    assert np.array_equal(lo, r1 - mid)
    assert np.array_equal(hi + (mid + lo), x)  # as whole_products puts it together
    assert (np.sign(mid) * np.sign(hi) >= 0).all() and (np.sign(lo) * np.sign(hi) >= 0).all()


# ---------------------------------------------------------------------------
# hash_rows.hip


def slots(K):
    blk, tpq = (1 if K <= 4 else 2), (2 if K == 2 else 1)

    def table(b, row):
        return 8 * b + (row >> 1) if K == 2 else 4 * (b // blk) + (row >> 2)

    def plane(b, row):
        return (row & 1) if K == 2 else 4 * (b % blk) + (row & 3)

    return blk, tpq, table, plane


@pytest.mark.parametrize("K", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("L", [1, 2, 3, 4, 5, 8, 9])
def test_slots_hold_every_plane_once_and_whole_tables_per_lane(K, L):
    blk, tpq, table, plane = slots(K)
    blocks = -(-L // (4 * tpq)) * blk
    held = Counter((table(b, row), plane(b, row)) for b in range(blocks) for row in range(16)
                   if table(b, row) < L and plane(b, row) < K)
    assert held == Counter((t, k) for t in range(L) for k in range(K))
    for b in range(0, blocks, blk):
        for g in range(4):
            for t in range(tpq):
                # Value 2 t + k of lane group g in the set: plane k of the table that
                # the gradient's select asks about.
                own = table(b, 4 * g + 2 * t)
                for k in range(K):
                    i = 2 * t + k
                    assert (table(b + i // 4, 4 * g + i % 4), plane(b + i // 4, 4 * g + i % 4)) == (own, k)


@pytest.mark.parametrize("NC", [1, 2, 4, 8, 16])
def test_chunk_exchange_follows_its_byte_offsets(NC):
    # exchange: permlane16_swap exchanges the odd 16-lane rows of its first
    # register with the even rows of the second, permlane32_swap the upper half
    # of the first with the lower half of the second.
    q = [[(g, c) for g in range(4)] for c in range(NC)]  # register c of lane group g: its own chunk c

    def swap16(a, b):
        for g in (0, 2):
            a[g + 1], b[g] = b[g], a[g + 1]

    def swap32(a, b):
        for g in (0, 1):
            a[g + 2], b[g] = b[g], a[g + 2]

    def exchange():
        if NC == 2:
            swap16(q[0], q[1])
        elif NC >= 4:
            for c in range(0, NC, 4):
                swap32(q[c], q[c + 2])
                swap32(q[c + 1], q[c + 3])
                swap16(q[c], q[c + 1])
                swap16(q[c + 2], q[c + 3])

    exchange()
    for i in range(NC):
        for g in range(4):
            owner = g if NC == 1 else ((g & 2) | i) if NC == 2 else (i & 3)
            chunk = 0 if NC == 1 else (g & 1) if NC == 2 else ((i & ~3) | g)
            assert q[i][g] == (owner, chunk)
    exchange()
    assert q == [[(g, c) for g in range(4)] for c in range(NC)]  # its own inverse


# ---------------------------------------------------------------------------
# narrow_causal.hip


@pytest.mark.parametrize("NE, ND", [(1, 1), (1, 4), (2, 2), (2, 4), (4, 2)])
def test_narrow_step_products(NE, ND):
    S, d = 16 * NE, 16 * ND
    rng = np.random.default_rng(NE + ND)
    K, V, W = rng.standard_normal((16, S)), rng.standard_normal((16, d)), rng.standard_normal((16, S))
    # B += K^T V from the row layout.
    B = [[zeros() for _ in range(ND)] for _ in range(NE)]
    for i in range(4):
        for e in range(NE):
            for f in range(ND):
                mfma([[K[4 * g + i, NE * lr + e]] for _, g, lr in LANES],
                     [[V[4 * g + i, ND * lr + f]] for _, g, lr in LANES], B[e][f])
    for e in range(NE):
        for f in range(ND):
            for lane, g, lr in LANES:
                for r in range(4):
                    s, c = 4 * NE * g + NE * r + e, ND * lr + f
                    np.testing.assert_allclose(B[e][f][lane][r], K[:, s] @ V[:, c], atol=1e-10)
    # P^T = K W^T from the quarter layout; (W B)^T with B as it stands; (P V)^T.
    P = zeros()
    for i in range(4 * NE):
        mfma([[K[lr, 4 * NE * g + i]] for _, g, lr in LANES], [[W[lr, 4 * NE * g + i]] for _, g, lr in LANES], P)
    for lane, g, lr in LANES:
        for r in range(4):
            P[lane][r] = P[lane][r] if 4 * g + r <= lr else 0.0
    o = [zeros() for _ in range(ND)]
    for r in range(4):
        for f in range(ND):
            for e in range(NE):
                mfma([[B[e][f][lane][r]] for lane, _, _ in LANES],
                     [[W[lr, 4 * NE * g + NE * r + e]] for _, g, lr in LANES], o[f])
            mfma([[V[4 * g + r, ND * lr + f]] for _, g, lr in LANES], [[P[lane][r]] for lane, _, _ in LANES], o[f])
    want = W @ (K.T @ V) + np.tril(W @ K.T) @ V
    for lane, g, lr in LANES:
        for m in range(ND):
            for i in range(4):
                got = o[(4 * m + i) % ND][lane][(4 * m + i) // ND]
                np.testing.assert_allclose(got, want[lr, 4 * ND * g + 4 * m + i], atol=1e-9)


# ---------------------------------------------------------------------------
# pack_heads.hip


@pytest.mark.parametrize("T, H, vec, launch", [(1, 3, 16, 1 << 23), (65, 5, 16, 1 << 23), (200, 12, 5, 7),
                                               (33, 1, 32, 2), (3, 17, 1, 4)])
def test_pack_heads_copies_every_chunk_once(T, H, vec, launch):
    # `launch`: workgroups of one launch (kPackLaunch), small here.
    B, tokens = 2, 1024 // vec
    shift = vec.bit_length() - 1 if vec & (vec - 1) == 0 else -1
    wgs = -(-T // tokens) * H
    written = {}
    for b in range(B):
        for first in range(0, wgs, launch):
            for block in range(min(wgs - first, launch)):
                wg = first + block
                h, t0 = wg % H, wg // H * tokens
                chunks = min(tokens, T - t0) * vec
                src, dst = ((b * T + t0) * H + h) * vec, ((b * H + h) * T + t0) * vec
                for c in range(chunks):
                    t = c >> shift if shift >= 0 else c // vec
                    assert dst + c not in written
                    written[dst + c] = src + t * H * vec + (c - t * vec)
    want = np.arange(B * T * H * vec).reshape(B, T, H, vec).transpose(0, 2, 1, 3).ravel()
    assert np.array_equal([written[i] for i in range(B * T * H * vec)], want)
