"""The small-batch kernels (prod_fwd_split / prod_bwd_split, 9 <= n <= 12; the
forward also at n = 8, one workgroup of 16 lanes per output block per row):
at the reference's published shapes (batch 1 .. 64) a row's partner loop is
split over the lanes of several workgroups and the partial blocks are summed in
LDS in a fixed order. Parity with the fp64 oracle for every op at n = 9, 10,
11, 12 (Euclidean, negative and null high generators), forced onto larger ragged
batches, against the whole-row kernels, and bitwise row independence.
Bar: normwise relative error <= 1e-5 for values and both gradients."""
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


def run(op, metric, a, b, gc):
    x = a.clone().requires_grad_()
    y = b.clone().requires_grad_()
    c = cc.products.product(op, x, y, metric)
    c.backward(gc)
    torch.cuda.synchronize()
    return c.detach(), x.grad, y.grad


def inputs(n, batch, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(batch, 1 << n, generator=g) for _ in range(3)]


METRICS = [(1,) * 10, (1,) * 6 + (-1, 1, -1, 1), (1,) * 9 + (0,), (-1,) * 4 + (1,) * 6 + (-1,),
           (1,) * 4 + (-1, 0, 1, 1, 1, 1, 1), (1,) * 9, (-1,) * 4 + (1, -1, 0, 1, 1)]


@pytest.mark.parametrize("metric", METRICS, ids=lambda m: "".join({1: "+", -1: "-", 0: "0"}[x] for x in m))
@pytest.mark.parametrize("op", O.OPS)
def test_small_batch_parity_n10_n11(op, metric):
    if op == "regressive" and 0 in metric:
        pytest.skip("regressive undefined for degenerate metrics")
    n = len(metric)
    for batch in (1, 3):
        a, b, gc = inputs(n, batch, 100 + batch)
        print(f"[case] small batch op={op} metric={metric} batch={batch}", flush=True)
        c, ga, gb = run(op, metric, a.cuda(), b.cuda(), gc.cuda())
        a64 = a.double().requires_grad_()
        b64 = b.double().requires_grad_()
        c64 = O.einsum_product(op, a64, b64, metric)
        c64.backward(gc.double())
        e = (rel_err(c, c64), rel_err(ga, a64.grad), rel_err(gb, b64.grad))
        assert max(e) <= TOL, e


@pytest.mark.parametrize("op", O.OPS)
def test_small_batch_parity_n12(op):
    metric = (1,) * 8 + (-1, 1, 1, -1)
    a, b, gc = inputs(12, 1, 120)
    print(f"[case] small batch n=12 op={op}", flush=True)
    c, ga, gb = run(op, metric, a.cuda(), b.cuda(), gc.cuda())
    a64 = a.double().requires_grad_()
    b64 = b.double().requires_grad_()
    c64 = O.einsum_product(op, a64, b64, metric)
    c64.backward(gc.double())
    e = (rel_err(c, c64), rel_err(ga, a64.grad), rel_err(gb, b64.grad))
    assert max(e) <= TOL, e


@pytest.mark.parametrize("op", O.OPS)
def test_split_forced_equals_whole_row_kernels(op, clf_env):
    """CLF_PRODUCT_PATH=split at a ragged batch of 300 rows (n = 10), 37 rows
    (n = 11) and 129 rows (n = 9) against the balanced / whole-row kernels (=blocked), which the
    oracle tests pin on their own. (CLF_GEOM_PATH=direct: the geometric product's
    matrix representations come before this switch.)"""
    clf_env.setenv("CLF_GEOM_PATH", "direct")
    for metric, batch in (((1,) * 8 + (-1, 1), 300), ((1,) * 11, 37), ((1,) * 5 + (-1, 1, 1, 1), 129)):
        n = len(metric)
        a, b, gc = [t.cuda() for t in inputs(n, batch, 130 + n)]
        print(f"[case] split forced op={op} n={n} batch={batch}", flush=True)
        clf_env.setenv("CLF_PRODUCT_PATH", "split")
        r_split = run(op, metric, a, b, gc)
        clf_env.setenv("CLF_PRODUCT_PATH", "blocked")
        r_blk = run(op, metric, a, b, gc)
        clf_env.delenv("CLF_PRODUCT_PATH")
        e = [rel_err(u, v) for u, v in zip(r_split, r_blk)]
        assert max(e) <= TOL, e


def test_split_rows_are_independent():
    """Rows computed in a batch of 21 equal, bit for bit, the same rows computed
    alone (both on the split kernels)."""
    metric = (1,) * 11
    a, b, gc = [t.cuda() for t in inputs(11, 21, 140)]
    full = run("lc", metric, a, b, gc)
    for r in (0, 7, 20):
        one = run("lc", metric, a[r:r + 1].contiguous(), b[r:r + 1].contiguous(), gc[r:r + 1].contiguous())
        for x, y in zip(full, one):
            assert torch.equal(x[r:r + 1], y)


METRICS8 = [(1,) * 8, (1,) * 6 + (-1, 1), (1,) * 7 + (0,), (-1,) * 4 + (1, -1, 0, 1), (1,) * 4 + (-1, 1, -1, -1)]


@pytest.mark.parametrize("metric", METRICS8, ids=lambda m: "".join({1: "+", -1: "-", 0: "0"}[x] for x in m))
@pytest.mark.parametrize("op", O.OPS)
def test_small_batch_forward_n8(op, metric, clf_env):
    """n = 8 forward at the published batches (1, 3, 64) against the fp64
    oracle, and forced onto the split kernel at a ragged batch of 129 rows
    against the whole-row kernels (=blocked)."""
    if op == "regressive" and 0 in metric:
        pytest.skip("regressive undefined for degenerate metrics")
    for batch in (1, 3, 64):
        a, b, _ = inputs(8, batch, 150 + batch)
        print(f"[case] small batch n=8 forward op={op} metric={metric} batch={batch}", flush=True)
        c = cc.products.product(op, a.cuda(), b.cuda(), metric)
        c64 = O.einsum_product(op, a.double(), b.double(), metric)
        assert rel_err(c, c64) <= TOL
    clf_env.setenv("CLF_GEOM_PATH", "direct")  # before the geometric product's matrix representations
    a, b, _ = [t.cuda() for t in inputs(8, 129, 158)]
    print(f"[case] split forced n=8 forward op={op} metric={metric} batch=129", flush=True)
    clf_env.setenv("CLF_PRODUCT_PATH", "split")
    c_split = cc.products.product(op, a, b, metric)
    clf_env.setenv("CLF_PRODUCT_PATH", "blocked")
    c_blk = cc.products.product(op, a, b, metric)
    clf_env.delenv("CLF_PRODUCT_PATH")
    assert rel_err(c_split, c_blk) <= TOL
