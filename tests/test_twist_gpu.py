"""The n = 8 geometric product one generator away from a real matrix algebra
(quaternionic type, one null generator): against the fp64 oracle for every sign
pattern class and place of the generator, and against the per-term kernels on a
larger batch, with a broadcast upstream gradient and with one gradient only."""
import pytest
import torch

import cliffordcuda_amd as cc
from oracle import clifford_oracle as O

pytestmark = pytest.mark.gpu
TOL = 1e-5  # normwise, as for every product: fp32 sums of 256 terms stay below 1e-6

SIGNATURES = [(1,) * 7 + (-1,), (-1,) + (1,) * 7, (1,) * 6 + (-1,) * 2, (1, -1, 1, 1, -1, 1, 1, 1),
              (-1,) * 5 + (1,) * 3, (1,) * 2 + (-1,) * 6,
              (1,) * 7 + (0,), (0,) + (1,) * 7, (1, 1, -1, 0, 1, -1, 1, 1), (-1,) * 7 + (0,),
              (1,) * 4 + (0,) + (-1,) * 3, (0, -1, 1, -1, 1, -1, 1, -1), (-1, 1, 1, -1, -1, 0, -1, -1)]


def ids(m):
    return "".join({1: "+", -1: "-", 0: "0"}[x] for x in m)


def rel_err(got, ref):
    got, ref = got.detach().double().cpu(), ref.detach().double().cpu()
    return float((got - ref).abs().max() / ref.abs().max())


def inputs(batch, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(batch, 256, generator=g) for _ in range(3)]


def gpu(metric, a, b, gc):
    x, y = a.cuda().requires_grad_(), b.cuda().requires_grad_()
    c = cc.geom_prod(x, y, metric)
    ga, gb = torch.autograd.grad(c, (x, y), gc)
    return c.detach(), ga, gb


@pytest.mark.parametrize("metric", SIGNATURES, ids=ids)
@pytest.mark.parametrize("batch", [1, 6, 17])
def test_against_oracle(metric, batch):
    a, b, gc = inputs(batch, 5 + batch)
    got = gpu(metric, a, b, gc.cuda())
    a64, b64 = a.double().requires_grad_(), b.double().requires_grad_()
    c64 = O.einsum_product("geom", a64, b64, metric)
    ref = (c64, *torch.autograd.grad(c64, (a64, b64), gc.double()))
    errs = [rel_err(u, v) for u, v in zip(got, ref)]
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("metric", [(1,) * 7 + (-1,), (1,) * 7 + (0,), (1, -1, 1, 1, -1, 1, 1, 1)], ids=ids)
def test_equals_per_term_kernels(metric, clf_env):
    a, b, gc = inputs(4099, 2)
    row = gc[:1].cuda().expand(4099, -1)
    got = gpu(metric, a, b, gc.cuda()) + gpu(metric, a, b, row)
    x, y = a.cuda().requires_grad_(), b.cuda().requires_grad_()
    ga, = torch.autograd.grad(cc.geom_prod(x, b.cuda(), metric), x, gc.cuda())
    gb, = torch.autograd.grad(cc.geom_prod(a.cuda(), y, metric), y, gc.cuda())
    assert torch.equal(ga, got[1]) and torch.equal(gb, got[2])
    clf_env.setenv("CLF_GEOM_PATH", "direct")
    ref = gpu(metric, a, b, gc.cuda()) + gpu(metric, a, b, row)
    clf_env.delenv("CLF_GEOM_PATH")
    errs = [rel_err(u, v) for u, v in zip(got, ref)]
    assert max(errs) <= TOL, errs
