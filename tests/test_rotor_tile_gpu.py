"""The rotor chain on tiles of generators (n = 9 .. 12) at the edges of a wave's
and a workgroup's rows: every row of a batch equals, bit for bit, the row as a
batch of its own (forward, x gradient, a broadcast upstream gradient), and the
bivector gradient is the sum of the rows' (rows past the end add nothing). The
values themselves are checked against the oracle in test_rotor_gpu.py."""
import pytest
import torch

import cliffordcuda_amd as cc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9, 10, 11, 12])
@pytest.mark.parametrize("batch", [2, 3, 5, 17])
def test_rows_alone_equal_rows_in_a_batch(n, batch):
    cl = cc.CliffordAlgebra([1] * n, device="cuda")
    g = torch.Generator().manual_seed(10 * n + batch)
    biv = (0.3 * torch.randn(1, n * (n - 1) // 2, generator=g)).cuda().requires_grad_()
    x = torch.randn(batch, 1 << n, generator=g).cuda().requires_grad_()
    gy = torch.randn(batch, 1 << n, generator=g).cuda()

    def step(rows, up):
        y = cl.apply_bivector(biv, rows)
        gb, gx = torch.autograd.grad(y, (biv, rows), up)
        return y.detach(), gx, gb

    y, gx, gb = step(x, gy)
    _, gx0, _ = step(x, gy[:1].expand(batch, -1))
    total = torch.zeros_like(gb, dtype=torch.float64)
    for r in range(batch):
        one = x[r:r + 1].detach().requires_grad_()
        y1, gx1, gb1 = step(one, gy[r:r + 1].contiguous())
        assert torch.equal(y[r:r + 1], y1) and torch.equal(gx[r:r + 1], gx1)
        assert torch.equal(gx0[r:r + 1], step(one, gy[:1].contiguous())[1])
        total += gb1.double()
    # the same fp32 statistics, summed in another order: 2^-23 times a few
    assert float((gb.double() - total).abs().max() / total.abs().max()) < 2e-6


@pytest.mark.parametrize("n,batch", [(9, 20011), (10, 9001), (11, 5003), (12, 4097)])
def test_bivector_gradient_over_many_row_groups(n, batch):
    """Past a resident grid a wave takes a second group of rows, its sums and its
    LDS carried over: the bivector gradient equals the fp64 sum of the gradients
    of pieces that no wave takes twice. The statistics are fp32 sums of the same
    products in another order: 2^-23 times a few, relative to the largest."""
    cl = cc.CliffordAlgebra([1] * n, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(n)
    biv = (0.3 * torch.randn(1, n * (n - 1) // 2, generator=g, device="cuda")).requires_grad_()
    x = torch.randn(batch, 1 << n, generator=g, device="cuda")
    # an upstream gradient along y's own change with the rotor: the sums do not cancel
    with torch.no_grad():
        gy = cl.apply_bivector(1.5 * biv, x)

    def gradient(rows, up):
        return torch.autograd.grad(cl.apply_bivector(biv, rows), (biv,), up)[0]

    total = torch.zeros_like(biv, dtype=torch.float64)
    for r in range(0, batch, 256):
        total += gradient(x[r:r + 256], gy[r:r + 256]).double()
    got = gradient(x, gy)
    print(f"[case] rotor many row groups n={n} batch={batch}", flush=True)
    assert float((got.double() - total).abs().max() / total.abs().max()) < 2e-6
