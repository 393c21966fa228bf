"""CPU model of the 32 x 32 geometric product (csrc/rep32.hip): the base / ext
decomposition with its gradients against the oracle, and the LDS layout."""
import itertools

import pytest
import torch

from oracle import clifford_oracle as O

BASE = 10


def popc(v):
    return bin(v).count("1")


def split(metric):
    """(ext generators, metric with the dummies), in the kernel's order of
    choice; None: not served."""
    n = len(metric)
    for d in range(3):
        k = n - BASE + d
        if k < 0 or k > 2 or (d == 2 and k != 1):
            continue
        for ext in sorted(itertools.combinations(range(n - 1, -1, -1), k), key=lambda e: tuple(-g for g in e)):
            base = [m for g, m in enumerate(metric) if g not in ext]
            for neg in range(d + 1):
                if 0 not in base and (sum(base) + d - 2 * neg) % 8 in (0, 2):
                    return sorted(ext), tuple(metric) + (-1,) * neg + (1,) * (d - neg)
    return None


def generators(squares):
    """Anticommuting real Pauli products P(x, z) on five qubits."""
    out, cand = [], [0] * BASE
    while len(out) < BASE:
        g = len(out)
        for c in range(cand[g] + 1, 1024):
            x, z = divmod(c, 32)
            if popc(x & z) % 2 == (squares[g] < 0) and all((popc(z & p) + popc(q & x)) % 2 for p, q in out):
                cand[g] = c
                out.append((x, z))
                if g + 1 < BASE:
                    cand[g + 1] = 0
                break
        else:
            out.pop()
    return out


def representation(metric, ext):
    """phi(e_I) for every base blade, with the blade's bit pattern."""
    base = [g for g in range(len(metric)) if g not in ext]
    gens = generators([metric[g] for g in base])
    mats = []
    for x, z in gens:
        m = torch.zeros(32, 32, dtype=torch.float64)
        for row in range(32):
            m[row, row ^ x] = (-1.0) ** popc(z & (row ^ x))
        mats.append(m)
    phi, blades = [torch.eye(32, dtype=torch.float64)], [0]
    for g, m in zip(base, mats):
        phi += [p @ m for p in phi]
        blades += [b | (1 << g) for b in blades]
    return torch.stack(phi), blades


@pytest.mark.parametrize("metric", [(1,) * 9 + (-1,), (1,) * 10 + (0,), (1, -1) * 5 + (-1,), (0,) + (1,) * 11,
                                    (-1,) * 3 + (1,) * 9, (1,) * 8 + (-1,), (1, 0) + (1,) * 7,
                                    (-1,) * 2 + (1,) * 7, (1,) * 8 + (-1,) * 2, (1,) * 8 + (-1,) * 3], ids=str)
def test_ext_products_and_gradients(metric):
    held = 1 << len(metric)  # the row's own coefficients; those with a dummy are zero
    ext, metric = split(metric)
    n = len(metric)
    phi, blades = representation(metric, ext)
    sigma = O.sign_value_table(n, metric).double()
    pats = [0]
    for g in ext:
        pats += [p | (1 << g) for p in pats]
    alpha = torch.tensor([(-1.0) ** popc(b) for b in blades], dtype=torch.float64)

    def blocks(x):  # coefficient of e_I e_S
        return [torch.stack([x[0, b | p] * float(sigma_e(b, p)) for b in blades]) for p in pats]

    euclid = O.sign_value_table(n, (1,) * n)

    def sigma_e(b, p):
        return euclid[b, p]

    def mat(v):
        return torch.einsum("i,irc->rc", v, phi)

    def row(ms):
        out = torch.zeros(1, 1 << n, dtype=torch.float64)
        for p, m in zip(pats, ms):
            v = torch.einsum("rc,irc->i", m, phi) / 32
            for b, c in zip(blades, v):
                out[0, b | p] = c * float(sigma_e(b, p))
        return out

    g = torch.Generator().manual_seed(1)
    a, b, gc = (torch.zeros(1, 1 << n, dtype=torch.float64) for _ in range(3))
    for t in (a, b, gc):
        t[:, :held] = torch.randn(1, held, generator=g, dtype=torch.float64)
        t.requires_grad_()
    A, B, G = ([mat(v.detach()) for v in blocks(t)] for t in (a, b, gc))
    Ah, Bh, Gh = ([mat(v.detach() * alpha) for v in blocks(t)] for t in (a, b, gc))
    S = range(len(pats))
    zero = torch.zeros(32, 32, dtype=torch.float64)
    C, GA, GB = ([zero.clone() for _ in S] for _ in range(3))
    for i in S:
        for j in S:
            s, odd = float(sigma[pats[i], pats[j]]), popc(i) & 1
            C[i ^ j] += s * A[i] @ (Bh if odd else B)[j]
            GA[i] += s * G[i ^ j] @ (Bh if odd else B)[j].T
            GB[j] += s * (Ah if odd else A)[i].T @ (Gh if odd else G)[i ^ j]
    c = O.einsum_product("geom", a, b, metric)
    ga, gb = torch.autograd.grad(c, (a, b), gc.detach())
    c = c.detach()
    for got, ref in ((row(C), c), (row(GA), ga), (row(GB), gb)):
        assert float((got - ref)[:, :held].abs().max() / ref.abs().max()) < 1e-12


def test_served_signatures():
    """Without null generators every signature at n = 9, 10, 11 and all but
    Cl(0, 12) at n = 12; at most n - 8 (n = 9), n - 9 or n - 10 null ones."""
    def served(n):
        return [q for q in range(n + 1) if split((1,) * (n - q) + (-1,) * q) is not None]
    assert [len(served(n)) for n in (9, 10, 11, 12)] == [10, 11, 12, 12]
    assert split((1,) * 8 + (0,)) is not None and split((1,) * 7 + (0, 0)) is None
    assert split((1,) * 10 + (0, 0))[0] == [10, 11] and split((1,) * 9 + (0,) * 3) is None


# one signature per (ext generators K, dummies D), low generators of both squares
FORMS = {(0, 1): (1, -1) + (1,) * 7, (1, 2): (1, -1, 1, 1, -1, 1, 1, 1, 1), (0, 0): (1, -1) * 5,
         (1, 1): (1, -1, 1, 1, -1) + (1,) * 5, (1, 0): (-1, 1) * 4 + (1, 1, -1), (2, 1): (1, -1, 1) * 3 + (1, 1),
         (2, 0): (1, 1, -1) * 4}


def test_forms():
    for (k, d), metric in FORMS.items():
        ext, dressed = split(metric)
        assert (len(ext), len(dressed) - len(metric)) == (k, d) and len(set(metric[:4])) == 2


def word(r, p):
    return ((r ^ ((r >> 3) & 1)) << 5) ^ (p ^ ((r & 7) << 2))


def test_lds_layout():
    """A bijection; the b32 column accesses of a half-wave touch 32 banks, eight
    lanes' b128 row writes eight groups, a b128 read set sixteen groups."""
    assert sorted(word(r, p) for r in range(32) for p in range(32)) == list(range(1024))
    for k in range(32):
        assert len({word(i ^ k, i) % 32 for i in range(32)}) == 32
        assert len({word(k ^ j, j) % 32 for j in range(32)}) == 32
    sets = [[0, 1, 2, 3, 12, 13, 14, 15, 20, 21, 22, 23, 24, 25, 26, 27],
            [4, 5, 6, 7, 8, 9, 10, 11, 16, 17, 18, 19, 28, 29, 30, 31]]
    for group in range(8):
        for x0 in range(0, 32, 8):
            assert len({word(x, 4 * group) // 4 % 8 for x in range(x0, x0 + 8)}) == 8
        for lanes in sets:
            assert len({word(x, 4 * group) // 4 % 16 for x in lanes}) == 16
