"""Products whose low four generators have different squares (or null ones):
against the fp64 oracle, values and both gradients, for every place of the odd
generator, a broadcast upstream gradient and one gradient alone; and against
the per-coefficient kernels."""
import pytest
import torch

import cliffordcuda_amd as cc
from oracle import clifford_oracle as O

pytestmark = pytest.mark.gpu
TOL = 1e-5  # normwise, as for every product: fp32 sums of at most 2^n terms stay below 1e-6
FN = {"geom": cc.geom_prod, "inner": cc.inner_prod, "lc": cc.left_contraction, "rc": cc.right_contraction}

METRICS = ["+-++", "0+++", "0000", "-0+-", "+++0-", "-+-+-", "00+-0", "+0+-+-", "++0-++", "-+++0++", "+-0-+0-",
           "0+++++++", "-+-+-0+0", "+-+-+-+-0"]


def signature(m):
    return tuple({"+": 1, "-": -1, "0": 0}[c] for c in m)


def rel_err(got, ref):
    got, ref = got.detach().double().cpu(), ref.detach().double().cpu()
    den = float(ref.abs().max())
    return float((got - ref).abs().max()) / (den if den > 0 else 1.0)


def grads(op, metric, a, b, gc):
    x, y = a.clone().requires_grad_(), b.clone().requires_grad_()
    c = FN[op](x, y, metric)
    return (c.detach(),) + torch.autograd.grad(c, (x, y), gc)


@pytest.mark.parametrize("op", list(FN))
@pytest.mark.parametrize("m", METRICS)
def test_against_oracle(op, m, clf_env):
    metric, n = signature(m), len(m)
    B = {4: 257, 5: 129, 6: 67, 7: 33, 8: 17}.get(n, 9)  # one row past the rows of a workgroup
    g = torch.Generator().manual_seed(n)
    a, b, gc = (torch.randn(B, 1 << n, generator=g) for _ in range(3))
    print(f"[case] mixed low op={op} metric={m} B={B}", flush=True)
    ad, bd, gd = a.cuda(), b.cuda(), gc.cuda()
    got = grads(op, metric, ad, bd, gd)
    a64, b64 = a.double().requires_grad_(), b.double().requires_grad_()
    c64 = O.einsum_product(op, a64, b64, metric)
    want = (c64,) + torch.autograd.grad(c64, (a64, b64), gc.double())
    for x, r in zip(got, want):
        assert rel_err(x, r) <= TOL
    one = grads(op, metric, ad, bd, gd[:1].expand(B, -1))
    x, y = ad.clone().requires_grad_(), bd.clone().requires_grad_()
    ga = torch.autograd.grad(FN[op](x, bd, metric), x, gd[:1].expand(B, -1).contiguous())[0]
    gb = torch.autograd.grad(FN[op](ad, y, metric), y, gd[:1].expand(B, -1).contiguous())[0]
    assert rel_err(one[1], ga) <= TOL and rel_err(one[2], gb) <= TOL
    clf_env.setenv("CLF_GEOM_PATH", "direct")
    clf_env.setenv("CLF_PRODUCT_PATH", "generic")
    for x, r in zip(got, grads(op, metric, ad, bd, gd)):
        assert rel_err(x, r) <= TOL


@pytest.mark.parametrize("op", list(FN))
@pytest.mark.parametrize("m", ["0+-+", "+0-00-+"])
def test_null_terms_are_passed_over(op, m, clf_env):
    """A term that a null generator takes away is not formed: an infinite
    coefficient reaches the same outputs as in the per-coefficient kernels."""
    metric = signature(m)
    g = torch.Generator().manual_seed(1)
    D = 1 << len(m)
    a, b, gc = (torch.randn(D, D, generator=g).cuda() for _ in range(3))
    a.diagonal().fill_(float("inf"))  # row r: coefficient r
    got = grads(op, metric, a, b, gc)
    clf_env.setenv("CLF_PRODUCT_PATH", "generic")
    for x, r in zip(got, grads(op, metric, a, b, gc)):
        assert torch.equal(x.isfinite(), r.isfinite())
