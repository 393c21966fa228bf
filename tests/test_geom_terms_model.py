"""CPU model of the term sums that the matrix-representation kernels give to rows
whose coefficients are not of one scale (csrc/geom_terms.h): the block form with
four generators of one square in front against the oracle, the signatures it has
to exist for, and the scale test's bound."""
import itertools
import random

import numpy as np
import pytest
import torch

from oracle import clifford_oracle as O


def popc(v):
    return bin(v).count("1")


def reorder(i, j):
    return sum(popc(i >> (b + 1)) for b in range(j.bit_length()) if (j >> b) & 1)


def four(metric):
    """(the four, ascending, their square), as the host picks them; None: no four."""
    sets = [[g for g, m in enumerate(metric) if m == s] for s in (1, -1)]
    for s, picks in zip((1, -1), sets):
        if picks[:4] == [0, 1, 2, 3]:
            return picks[:4], s
    for s, picks in zip((1, -1), sets):
        if len(picks) >= 4:
            return picks[:4], s
    return None


def block_products(metric, a, b, gc):
    """c, ga, gb of one row from blocks, with the kernel's signs and places."""
    n = len(metric)
    c4, square = four(metric)
    rest = [g for g in range(n) if g not in c4]
    neg = sum(1 << k for k, g in enumerate(rest) if metric[g] < 0)
    nul = sum(1 << k for k, g in enumerate(rest) if metric[g] == 0)
    nb = 1 << (n - 4)

    def place(h):
        for c in c4:
            below = h & ((1 << c) - 1)
            h = below | ((h ^ below) << 1)
        return h

    def chi(h):
        return [popc(place(h) & ((1 << c) - 1)) & 1 for c in c4]

    offset = [sum(((l >> k) & 1) << c for k, c in enumerate(c4)) for l in range(16)]
    odd = [popc(l) & 1 for l in range(16)]

    def block(row, h):
        m = chi(h)
        sign = [(-1.0) ** sum(m[k] for k in range(4) if (l >> k) & 1) for l in range(16)]
        return np.array([row[place(h) | offset[l]] * sign[l] for l in range(16)])

    def store(out, h, acc):
        m = chi(h)
        for l in range(16):
            out[place(h) | offset[l]] = acc[l] * (-1.0) ** sum(m[k] for k in range(4) if (l >> k) & 1)

    low = [[(-1.0) ** (reorder(i, j) + (popc(i & j) if square < 0 else 0)) for j in range(16)] for i in range(16)]
    alt = np.array([(-1.0) ** o for o in odd])
    outs = [np.zeros(1 << n) for _ in range(3)]
    for h in range(nb):
        accs = [np.zeros(16) for _ in range(3)]
        for m in range(nb):
            for mode, (x, y) in enumerate(((a, b), (b, gc), (a, gc))):
                i, j = ((m, m ^ h), (h, m), (m, h))[mode]
                if i & j & nul:
                    continue
                s = (-1.0) ** (reorder(i, j) + popc(i & j & neg))
                u, v = block(x, m), block(y, m ^ h)
                flip = alt if popc(i) & 1 else np.ones(16)
                if mode == 0:
                    v = v * s * flip
                else:
                    u = u * s * flip
                if mode == 2:
                    v = v * flip
                for il, jl in itertools.product(range(16), range(16)):
                    t = low[il][jl]
                    if mode == 0:
                        accs[0][il ^ jl] += t * u[il] * v[jl]
                    elif mode == 1:
                        accs[1][il] += t * u[jl] * v[il ^ jl]
                    else:
                        accs[2][jl] += t * u[il] * v[il ^ jl]
        for out, acc in zip(outs, accs):
            store(out, h, acc)
    return outs


@pytest.mark.parametrize("m", ["++++", "-----", "+-+-+-+", "-++0-+++", "0++--++-", "-+-+-+-+", "++0-+-0+"])
def test_blocks_against_oracle(m):
    metric = tuple({"+": 1, "-": -1, "0": 0}[c] for c in m)
    n = len(m)
    g = torch.Generator().manual_seed(n)
    a, b, gc = (torch.randn(1, 1 << n, generator=g, dtype=torch.float64).requires_grad_() for _ in range(3))
    c = O.einsum_product("geom", a, b, metric)
    ga, gb = torch.autograd.grad(c, (a, b), gc.detach())
    got = block_products(metric, *(t.detach()[0].numpy() for t in (a, b, gc)))
    for u, v in zip(got, (c.detach(), ga, gb)):
        assert np.abs(u - v[0].numpy()).max() < 1e-12 * np.abs(v[0].numpy()).max()


def test_four_of_one_square():
    """Wherever a representation is used: n = 7 without null generators, n = 8
    with at most one, n = 9 .. 12 with at most two."""
    for n, most in ((7, 0), (8, 1), (9, 1), (10, 1), (11, 2), (12, 2)):
        for nul in range(most + 1):
            for q in range(n - nul + 1):
                assert max(q, n - nul - q) >= 4
                metric = [0] * nul + [-1] * q + [1] * (n - nul - q)
                random.Random(n).shuffle(metric)
                assert four(tuple(metric)) is not None


def one_scale(x):
    q = float((x.astype(np.float32) ** 2).sum())
    return 2.0 ** -80 <= q <= 2.0 ** 80 and 8 * int((np.abs(x) >= np.sqrt(q / x.size) / 4).sum()) >= 5 * x.size


def test_scale_bound():
    """Two rows that pass have, for every coefficient, a sum of |terms| of at
    least N r_a r_b / 64; N(0, 1) and uniform rows pass, graded ones do not."""
    rng = np.random.default_rng(3)
    N = 256
    k = np.arange(N)
    worst = []
    for share in (0.63, 0.7, 0.8, 1.0):
        for _ in range(40):
            rows = []
            for _ in range(2):
                x = rng.standard_normal(N) * 1e-4
                keep = rng.permutation(N)[:int(np.ceil(share * N))]
                x[keep] = rng.choice([0.3, 1.0, 1.2], keep.size) * rng.choice([-1, 1], keep.size)
                rows.append(x)
            if not all(one_scale(x) for x in rows):
                continue
            a, b = (np.abs(x) for x in rows)
            terms = np.array([(a * b[k ^ c]).sum() for c in range(N)])
            ra, rb = (np.sqrt((x ** 2).mean()) for x in rows)
            worst.append(terms.min() / (N * ra * rb))
    assert len(worst) > 100 and min(worst) >= 1 / 64
    assert all(one_scale(rng.standard_normal(N)) and one_scale(rng.uniform(-1, 1, N)) for _ in range(2000))
    grade = np.array([popc(i) for i in range(N)])
    assert not one_scale(rng.standard_normal(N) * 10.0 ** -grade)
    assert not one_scale(rng.standard_normal(N) * (grade == 1))
    assert not one_scale(np.where(grade == 0, np.inf, 1.0)) and not one_scale(np.full(N, np.nan))
