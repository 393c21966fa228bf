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


def sums(metric, x, y, which):
    """In fp64, the value and the sum of the |terms| of c (x = a, y = b), ga
    (x = b, y = gc) or gb (x = a, y = gc), with the oracle's signs."""
    n = len(metric)
    sigma = O.sign_value_table(n, metric).cuda().double()
    k = torch.arange(1 << n, device="cuda")
    x, y = x.cuda().double(), y.cuda().double()
    out, terms = torch.zeros_like(y), torch.zeros_like(y)
    for i in range(1 << n):
        s = sigma[i, i ^ k] if which == "c" else sigma[k, i] if which == "ga" else sigma[i, k]
        t = x[:, i:i + 1] * y[:, i ^ k] * s
        out += t
        terms += t.abs()
    return out, terms


def worst(got, ref, terms, scale=1.0):
    """Largest error over the bar."""
    err = (got.double() - ref).abs()
    assert bool((err[terms == 0] == 0).all())  # no term: an exact zero
    n = got.shape[-1].bit_length() - 1
    return float((err / terms.clamp_min(1e-300)).max()) / (scale * bar(n))


def check(metric, a, b, gc):
    ad, bd = a.cuda().requires_grad_(), b.cuda().requires_grad_()
    c = cc.geom_prod(ad, bd, metric)
    got = (c.detach(), *torch.autograd.grad(c, (ad, bd), gc.cuda()))
    want = (sums(metric, a, b, "c"), sums(metric, b, gc, "ga"), sums(metric, a, gc, "gb"))
    return [worst(u, *v) for u, v in zip(got, want)]


PAIRS = [("graded", "graded", "dense"), ("near one", "near one", "near one"), ("vector", "vector", "vector"),
         ("dense", "large vector", "dense"), ("share 0.55", "share 0.66", "dense"),
         ("share 0.8", "share 0.85", "share 0.8"), ("dense", "dense", "dense"), ("tiny", "dense", "tiny")]


FEW = {8: 19, 9: 771, 10: 131, 11: 35, 12: 9}  # past the rows that the per-term kernels keep
MANY = {8: 1031, 9: 2100, 10: 2100, 11: 1050, 12: 520}  # one workgroup a row


@pytest.mark.parametrize("m", SIGNATURES)
def test_error_against_the_terms(m):
    metric, n = signature(m), len(m)
    for kinds in PAIRS:
        g = torch.Generator().manual_seed(n)
        count = (MANY if kinds[0] == "graded" else FEW)[n]
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
    count = {8: 37, 9: 800, 10: 140, 11: 40}[n]
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
        W = w.expand(count, -1)
        want = (sums(metric, *((x, W) if side == 0 else (W, x)), "c"), sums(metric, W, gy, "ga" if side == 0 else "gb"),
                [t.sum(0, keepdim=True) for t in sums(metric, x, gy, "gb" if side == 0 else "ga")])
        errs = [worst(u, *v, scale) for u, v, scale in zip(got, want, (1, 1, count ** 0.5))]
        assert max(errs) <= 1, (kinds, errs)
