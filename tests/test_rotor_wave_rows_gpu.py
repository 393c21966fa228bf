"""The rotor chain at n = 9 .. 12 (tiles of generators) on a few rows and on a
batch of many workgroups: the same rows equal, bit for bit, whatever batch they
come in (the order of a row's planes depends on n alone), and both equal the fp64
oracle chain within 1e-5. Forward and transposed (the x gradient through a rotor
that needs no gradient)."""
import pytest
import torch

import cliffordcuda_amd as cc
from oracle import clifford_oracle as O

pytestmark = pytest.mark.gpu
TOL = 1e-5


def rel_err(got, ref):
    got = got.detach().double().cpu()
    ref = ref.detach().double().cpu()
    den = float(ref.abs().max())
    return float((got - ref).abs().max()) / (den if den > 0 else 1.0)


@pytest.mark.parametrize("n,B", [(9, 12300), (10, 1100), (11, 1100), (12, 1100)])
def test_chain_on_few_and_many_rows(n, B):
    cl = cc.CliffordAlgebra([1] * (n - 1) + [-1], device="cuda")
    g = torch.Generator().manual_seed(40 + n)
    biv = (0.3 * torch.randn(1, n * (n - 1) // 2, generator=g)).cuda()
    x = torch.randn(B, 1 << n, generator=g).cuda()
    gy = torch.randn(B, 1 << n, generator=g).cuda()
    rows = torch.tensor([0, 1, 517, B - 1], device="cuda")
    print(f"[case] rotor few and many rows n={n} B={B}", flush=True)
    with torch.no_grad():
        cs = cl.compile_bivector(biv)
        y_big = cl.apply_rotor(cs, x)
        y_small = cl.apply_rotor(cs, x[rows].contiguous())
    assert torch.equal(y_big[rows], y_small)
    xb = x.clone().requires_grad_()
    (gx_big,) = torch.autograd.grad(cl.apply_rotor(cs, xb), (xb,), gy)
    xs = x[rows].clone().requires_grad_()
    (gx_small,) = torch.autograd.grad(cl.apply_rotor(cs, xs), (xs,), gy[rows].contiguous())
    assert torch.equal(gx_big[rows], gx_small)
    cs64 = cs.detach().double().cpu()
    x64 = x[rows].double().cpu().requires_grad_()
    y64 = O.givens_chain_apply(cs64, x64, n)
    (gx64,) = torch.autograd.grad(y64, (x64,), gy[rows].double().cpu())
    assert rel_err(y_small, y64) <= TOL
    assert rel_err(gx_small, gx64) <= TOL
