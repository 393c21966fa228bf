"""The geometric product of large algebras on 32 x 32 matrices: against the
fp64 oracle at the edges of a workgroup's rows, in every form, and against the per-term
kernels over every form the rule accepts (signs in any order, ext generators of
each square, a broadcast upstream gradient, one gradient only)."""
import pytest
import torch

import cliffordcuda_amd as cc
from oracle import clifford_oracle as O
from tests.test_rep32_model import FORMS

pytestmark = pytest.mark.gpu
TOL = 1e-5  # normwise, as for every product: 3 sqrt(2^n) sums of fp32 terms stay below 1e-6

SIGNATURES = [
    (1,) * 8 + (-1,), (1, -1, 1, -1, 1, 1, 1, 1, -1), (-1, 1) + (1,) * 6 + (-1,), (1,) * 8 + (0,), (0,) + (-1, 1) * 4,
    (1,) * 8 + (-1,) * 2, (1, 0) + (1,) * 8, (-1,) * 10, (1,) * 8 + (-1,) * 3, (1, -1, 1) * 3 + (0, 0),  # with dummies
    (1,) * 10, (1,) * 9 + (-1,), (-1,) * 4 + (1,) * 6, (1, -1) * 5, (-1,) * 9 + (1,),  # n = 10, real type
    (1,) * 11, (1,) * 10 + (-1,), (1,) * 10 + (0,), (0,) + (1,) * 10, (-1, 1) * 4 + (1, 1, -1),
    (1,) * 5 + (0,) + (-1,) * 5,
    (1,) * 12, (1,) * 11 + (-1,), (1,) * 9 + (-1,) * 3, (1,) * 10 + (0, 0), (0, -1) + (1,) * 10,
    (1, 1, -1) * 4, (-1,) * 11 + (1,),
]


def ids(m):
    return "".join({1: "+", -1: "-", 0: "0"}[x] for x in m)


def rel_err(got, ref):
    got, ref = got.detach().double().cpu(), ref.detach().double().cpu()
    return float((got - ref).abs().max() / ref.abs().max())


def inputs(batch, n, seed, count=3):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(batch, 1 << n, generator=g) for _ in range(count)]


def gpu(metric, a, b, gc):
    x, y = a.cuda().requires_grad_(), b.cuda().requires_grad_()
    c = cc.geom_prod(x, y, metric)
    ga, gb = torch.autograd.grad(c, (x, y), gc)
    return c.detach(), ga, gb


# FORMS: one signature per (K, D) whose low generators have both squares, so that
# no few rows go to the per-term kernels; of the others those with K > 0 do
@pytest.mark.parametrize("metric", list(FORMS.values()) + [
    (1,) * 8 + (-1,), (-1,) * 2 + (1,) * 7, (1,) * 10, (1,) * 8 + (-1,) * 2, (1,) * 10 + (-1,), (1,) * 8 + (-1,) * 3,
    (1,) * 12], ids=ids)
@pytest.mark.parametrize("batch", [1, 3, 5])
def test_against_oracle(metric, batch):
    a, b, gc = inputs(batch, len(metric), 3 + batch)
    got = gpu(metric, a, b, gc.cuda())
    a64, b64 = a.double().requires_grad_(), b.double().requires_grad_()
    c64 = O.einsum_product("geom", a64, b64, metric)
    ref = (c64, *torch.autograd.grad(c64, (a64, b64), gc.double()))
    errs = [rel_err(u, v) for u, v in zip(got, ref)]
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("metric", SIGNATURES, ids=ids)
def test_equals_per_term_kernels(metric, clf_env):
    rows = 771 if len(metric) == 9 else 131 if len(metric) == 10 else 33 + len(metric)  # past the few-rows rule
    a, b, gc = inputs(rows, len(metric), 7)
    row = gc[:1].cuda().expand(rows, -1)  # the gradient of a weighted sum: batch stride 0
    got = gpu(metric, a, b, gc.cuda()) + gpu(metric, a, b, row)
    x, y = a.cuda().requires_grad_(), b.cuda().requires_grad_()
    ga, = torch.autograd.grad(cc.geom_prod(x, b.cuda(), metric), x, gc.cuda())
    gb, = torch.autograd.grad(cc.geom_prod(a.cuda(), y, metric), y, gc.cuda())
    assert torch.equal(ga, got[1]) and torch.equal(gb, got[2])  # one gradient only: the same bits
    clf_env.setenv("CLF_GEOM_PATH", "direct")
    ref = gpu(metric, a, b, gc.cuda()) + gpu(metric, a, b, row)
    clf_env.delenv("CLF_GEOM_PATH")
    errs = [rel_err(u, v) for u, v in zip(got, ref)]
    assert max(errs) <= TOL, errs
