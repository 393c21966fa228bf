"""The geometric product on rows whose coefficients are not of one scale, where a
matrix representation would round against the norm of the whole row: graded
rows, rows near 1, vectors, sparse rows, infinities and NaN. Every coefficient is
compared with the fp64 sum of its terms, its error measured against the sum of
their absolute values.

Bar: a chain of 2^n fp32 multiply-adds, each rounding at most 2^-24 of a partial
sum that the sum of |terms| bounds, taken as independent: 4 sqrt(2^n) 2^-24
(7.6e-6 at n = 10; the worst case, 2^n 2^-24, is 8 to 16 times that)."""
import pytest
import torch

import cliffordcuda_amd as cc
from oracle import clifford_oracle as O

pytestmark = pytest.mark.gpu

SIGNATURES = ["+" * 7 + "-", "-+-+++++", "+" * 7 + "0", "0" + "+" * 7, "+-0++-++", "-+-+-+-0", "-" * 7 + "0",  # n = 8
              "+" * 8 + "-", "+-+-+-+++", "+" * 7 + "--", "0" + "+" * 8, "+" * 10, "+-" * 5, "+" * 8 + "--",
              "0" + "+" * 9, "-+-+-+-+-+-", "+" * 10 + "-", "+" * 8 + "---", "+" * 10 + "0", "0+-+-+-+-+-+", "+" * 12]


def signature(m):
    return tuple({"+": 1, "-": -1, "0": 0}[c] for c in m)


def bar(n):
    return 4 * 2 ** (n / 2) * 2.0 ** -24


def rows(kind, n, count, gen):
    """Rows of one kind, (count, 2^n)."""
    grade = O.grades(n)
    x = torch.randn(count, 1 << n, generator=gen)
    if kind == "graded":
        return x * 10.0 ** -grade.float()
    if kind == "near one":
        x = x * (grade == 2) * 1e-3
        x[:, 0] = 1
        return x
    if kind == "vector":
        return x * (grade == 1)
    if kind == "large vector":  # beside small other coefficients
        return torch.where(grade == 1, 1e6 * x, x)
    if kind.startswith("share"):  # a share of the coefficients is there
        keep = torch.rand(count, 1 << n, generator=gen) < float(kind.split()[1])
        return x * keep
    if kind == "tiny":
        return x * 1e-18
    assert kind == "dense"
    return x


def term_sums(metric, x, y, which):
    """Sums of the |terms| of c (x = a, y = b), ga (x = b, y = gc), gb (x = a, y = gc)."""
    n = len(metric)
    nul = sum(1 << g for g, m in enumerate(metric) if m == 0)
    k = torch.arange(1 << n, device="cuda")
    x, y = x.abs().double(), y.abs().double()
    out = torch.zeros_like(x)
    for i in range(1 << n):
        other = i ^ k
        hit = (i & (other if which == "c" else k) & nul) == 0
        out += x[:, i:i + 1] * y[:, other] * hit
    return out


def check(metric, a, b, gc):
    """Largest error of c, ga, gb over the bar."""
    n = len(metric)
    ad, bd = a.cuda().requires_grad_(), b.cuda().requires_grad_()
    c = cc.geom_prod(ad, bd, metric)
    got = (c.detach(), *torch.autograd.grad(c, (ad, bd), gc.cuda()))
    a64, b64 = a.double().requires_grad_(), b.double().requires_grad_()
    c64 = O.einsum_product("geom", a64, b64, metric)
    ref = (c64.detach(), *torch.autograd.grad(c64, (a64, b64), gc.double()))
    terms = (term_sums(metric, a.cuda(), b.cuda(), "c"), term_sums(metric, b.cuda(), gc.cuda(), "ga"),
             term_sums(metric, a.cuda(), gc.cuda(), "gb"))
    worst = []
    for u, v, t in zip(got, ref, terms):
        err = (u.double() - v.cuda()).abs()
        assert bool((err[t == 0] == 0).all())  # no term: an exact zero
        worst.append(float((err / t.clamp_min(1e-300)).max()) / bar(n))
    return worst


PAIRS = [("graded", "graded", "dense"), ("near one", "near one", "near one"), ("vector", "vector", "vector"),
         ("dense", "large vector", "dense"), ("share 0.55", "share 0.66", "dense"),
         ("share 0.8", "share 0.85", "share 0.8"), ("dense", "dense", "dense"), ("tiny", "dense", "tiny")]


@pytest.mark.parametrize("m", SIGNATURES)
def test_error_against_the_terms(m):
    metric, n = signature(m), len(m)
    for kinds in PAIRS:
        g = torch.Generator().manual_seed(n)
        count = {8: 19, 9: 515, 10: 131, 11: 35, 12: 5}[n] if kinds[0] == "graded" else 5  # past the few-rows rule
        a, b, gc = (rows(k, n, count, g) for k in kinds)
        print(f"[case] scales {m} {kinds} rows={count}", flush=True)
        assert max(check(metric, a, b, gc)) <= 1, kinds


@pytest.mark.parametrize("m", ["+" * 7 + "-", "+" * 7 + "0", "+-+-+-+++", "+" * 10, "-+-+-+-+-+-", "+" * 12])
def test_rows_do_not_depend_on_their_neighbours(m):
    """Rows of one scale between others: the bits of the same rows alone."""
    metric, n = signature(m), len(m)
    count = {8: 53, 9: 1031, 10: 261, 11: 67, 12: 21}[n]
    g = torch.Generator().manual_seed(2)
    a, b, gc = (rows("dense", n, count, g) for _ in range(3))
    odd = torch.arange(count) % 3 == 1
    mixed = [torch.where(odd[:, None], rows("graded", n, count, g), t) for t in (a, b, gc)]

    def run(a, b, gc):
        x, y = a.cuda().requires_grad_(), b.cuda().requires_grad_()
        c = cc.geom_prod(x, y, metric)
        return (c.detach(), *torch.autograd.grad(c, (x, y), gc.cuda()))

    for u, v in zip(run(a, b, gc), run(*mixed)):
        assert torch.equal(u[~odd], v[~odd])


@pytest.mark.parametrize("m", ["+" * 7 + "-", "+" * 7 + "0", "+-0++-++", "+" * 8 + "-", "0" + "+" * 8, "+" * 10, "+-" * 5, "0" + "+" * 9, "+-+-+-+-+-0"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_not_finite(m, value, clf_env):
    """An infinite or undefined coefficient reaches the coefficients it
    multiplies and no others, as on the per-term kernels."""
    metric, n = signature(m), len(m)
    count = {8: 37, 9: 600, 10: 140, 11: 40}[n]
    g = torch.Generator().manual_seed(4)
    a, b, gc = (rows("dense", n, count, g) for _ in range(3))
    b[:, ::2] = 0  # inf * 0 and inf * x
    at = torch.arange(count)
    a[at[::2], (37 * at[::2]) % (1 << n)] = value
    gc[at[1::4], (11 * at[1::4]) % (1 << n)] = value

    def run():
        x, y = a.cuda().requires_grad_(), b.cuda().requires_grad_()
        c = cc.geom_prod(x, y, metric)
        return (c.detach(), *torch.autograd.grad(c, (x, y), gc.cuda()))

    got = run()
    clf_env.setenv("CLF_GEOM_PATH", "direct")
    for u, v in zip(got, run()):
        assert torch.equal(u.isnan(), v.isnan()) and torch.equal(u.isinf(), v.isinf())
        assert torch.equal(u[u.isinf()], v[v.isinf()])


@pytest.mark.parametrize("m", ["+" * 7, "+" * 6 + "-", "-+-+-+-", "+" * 7 + "-", "+" * 9, "+-" * 4 + "+", "+" * 8 + "-",
                               "+" * 9 + "0", "-+" * 4 + "+0", "+" * 10])
@pytest.mark.parametrize("side", [0, 1])
def test_layers(m, side):
    """A layer's value and gradients (weight one row of the batch's products):
    the weight gradient sums batch * 2^n terms, the bar grows with their root."""
    metric, n = signature(m), len(m)
    count = 37
    for kinds in (("graded", "near one", "dense"), ("vector", "dense", "near one"), ("share 0.6", "share 0.9", "dense"),
                  ("dense", "dense", "graded"), ("dense", "dense", "dense")):
        g = torch.Generator().manual_seed(n)
        x, w, gy = rows(kinds[0], n, count, g), rows(kinds[1], n, 1, g), rows(kinds[2], n, count, g)
        print(f"[case] layer scales {m} side={side} {kinds}", flush=True)
        xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
        y = cc.bcast.bcast_product("geom", xd, wd, metric, side=side)
        got = (y.detach(), *torch.autograd.grad(y, (xd, wd), gy.cuda()))
        x64, w64 = x.double().requires_grad_(), w.double().requires_grad_()
        a64, b64 = (x64, w64.expand_as(x64)) if side == 0 else (w64.expand_as(x64), x64)
        y64 = O.einsum_product("geom", a64, b64, metric)
        ref = (y64.detach(), *torch.autograd.grad(y64, (x64, w64), gy.double()))
        X, W, G = x.cuda(), w.cuda().expand(count, -1), gy.cuda()
        terms = (term_sums(metric, *((X, W) if side == 0 else (W, X)), "c"),
                 term_sums(metric, W, G, "ga" if side == 0 else "gb"),
                 term_sums(metric, X, G, "gb" if side == 0 else "ga").sum(0, keepdim=True))
        for u, v, t, scale in zip(got, ref, terms, (1, 1, count ** 0.5)):
            err = (u.double() - v.cuda()).abs()
            assert bool((err[t == 0] == 0).all())
            assert float((err / t.clamp_min(1e-300)).max()) <= scale * bar(n), kinds
