"""GPU parity of the product layers (broadcast weight, MFMA GEMM path for
7 <= n <= 10) against the oracle, and against the per-row kernels on the
expanded weight at the full C3 size."""
import pytest
import torch

import cliffordcuda_amd as cc
from cliffordcuda_amd import bcast
from oracle import clifford_oracle as O

pytestmark = pytest.mark.gpu
TOL = 1e-5


def rel_err(got, ref):
    got = got.detach().double().cpu()
    ref = ref.detach().double().cpu()
    den = float(ref.abs().max())
    return float((got - ref).abs().max()) / (den if den > 0 else 1.0)


LAYERS = [("geom", cc.GeometricProductLayer), ("wedge", cc.WedgeProductLayer), ("inner", cc.InnerProductLayer),
          ("lc", cc.LeftContractionLayer), ("rc", cc.RightContractionLayer),
          ("regressive", cc.RegressiveProductLayer)]


@pytest.mark.parametrize("metric", [(1,) * 7, (1,) * 7 + (-1,), (1,) * 6 + (-1, 0), (-1, 1) * 4, (1,) * 9 + (0,),
                                    (1, 1, 1, 1, 1)],
                         ids=lambda m: "".join({1: "+", -1: "-", 0: "0"}[x] for x in m))
@pytest.mark.parametrize("op,cls", LAYERS, ids=[l[0] for l in LAYERS])
def test_layer_parity(op, cls, metric):
    if op == "regressive" and 0 in metric:
        pytest.skip("regressive undefined for degenerate metrics")
    n = len(metric)
    cl = cc.CliffordAlgebra(metric, device="cuda")
    layer = cls(cl)
    g = torch.Generator().manual_seed(3)
    B = 300 if n < 10 else 40
    x = torch.randn(B, 1 << n, generator=g)
    w = 0.25 * torch.randn(1, 1 << n, generator=g)
    gy = torch.randn(B, 1 << n, generator=g)
    with torch.no_grad():
        layer.weight.copy_(w.cuda())
    xd = x.cuda().requires_grad_()
    print(f"[case] layer op={op} metric={metric}", flush=True)
    y = layer(xd)
    y.backward(gy.cuda())
    x64 = x.double().requires_grad_()
    w64 = w.double().requires_grad_()
    y64 = O.layer_forward(op, x64, w64, metric)
    y64.backward(gy.double())
    assert rel_err(y, y64) <= TOL
    assert rel_err(xd.grad, x64.grad) <= TOL
    assert rel_err(layer.weight.grad, w64.grad) <= TOL


@pytest.mark.parametrize("op", ["geom", "lc", "regressive"])
def test_weight_on_left(op):
    metric = (1,) * 7 + (-1,)
    g = torch.Generator().manual_seed(4)
    x = torch.randn(130, 256, generator=g)
    w = torch.randn(1, 256, generator=g)
    gy = torch.randn(130, 256, generator=g)
    xd = x.cuda().requires_grad_()
    wd = w.cuda().requires_grad_()
    y = bcast.bcast_product(op, xd, wd, metric, side=1)
    y.backward(gy.cuda())
    x64 = x.double().requires_grad_()
    w64 = w.double().requires_grad_()
    y64 = O.einsum_product(op, w64.expand_as(x64), x64, metric)
    y64.backward(gy.double())
    assert rel_err(y, y64) <= TOL
    assert rel_err(xd.grad, x64.grad) <= TOL
    assert rel_err(wd.grad, w64.grad) <= TOL


def test_c3_full_batch_vs_per_row_kernels(clf_env):
    """GeometricProductLayer Cl(8,0), x (262144, 256) ~ N(0,1),
    w ~ N(0, 1/16). Three independent HIP algorithms agree at the full batch,
    values and both gradients: the matrix-representation layer kernels (the
    path Cl(8,0) takes), the MFMA GEMM against the weight's 256 x 256 matrix,
    and the per-term product kernels on the expanded weight (both forced with
    CLF_GEOM_PATH=direct); a row sample also matches the oracle."""
    cl = cc.CliffordAlgebra([1] * 8, device="cuda")
    layer = cc.GeometricProductLayer(cl)
    g = torch.Generator().manual_seed(0)
    B = 262144
    x = torch.randn(B, 256, generator=g)
    w = 0.25 * torch.randn(1, 256, generator=g)
    with torch.no_grad():
        layer.weight.copy_(w.cuda())

    def run_layer():
        layer.weight.grad = None
        xd = x.cuda().requires_grad_()
        y = layer(xd)
        y.sum().backward()
        return y.detach(), xd.grad, layer.weight.grad.clone()

    y, gx, gw = run_layer()
    clf_env.setenv("CLF_GEOM_PATH", "direct")
    y1, gx1, gw1 = run_layer()
    x2 = x.cuda().requires_grad_()
    w2 = w.cuda().requires_grad_()
    y2 = cc.geom_prod(x2, w2.expand(B, 256).contiguous())
    y2.sum().backward()
    clf_env.delenv("CLF_GEOM_PATH")
    for a, b, c in ((y, y1, y2), (gx, gx1, x2.grad), (gw, gw1, w2.grad)):
        assert rel_err(a, b) <= TOL
        assert rel_err(b, c) <= TOL
    rows = torch.tensor([0, 5, 123456, B - 1])
    y64 = O.layer_forward("geom", x[rows].double(), w.double())
    assert rel_err(y[rows.cuda()], y64) <= TOL


def test_c3_full_batch_gradients_vs_oracle_batch_sum():
    """BASELINE config C3 at its full batch against the fp64 oracle, both
    gradients. With the upstream gradient all ones and the layer linear in x,
    L = sum_b sum_k (x_b w)_k = sum_k (S w)_k with S = sum_b x_b (fp64), so
    the full-batch weight gradient equals the oracle's gradient on the single
    row S, and every row of the x gradient equals the oracle's x gradient of
    one row (it does not depend on x). The forward is checked through the
    same linearity: sum_b y_b = S w."""
    cl = cc.CliffordAlgebra([1] * 8, device="cuda")
    layer = cc.GeometricProductLayer(cl)
    g = torch.Generator().manual_seed(0)
    B = 262144
    x = torch.randn(B, 256, generator=g)
    w = 0.25 * torch.randn(1, 256, generator=g)
    with torch.no_grad():
        layer.weight.copy_(w.cuda())
    xd = x.cuda().requires_grad_()
    print(f"[case] C3 full batch B={B} batch-sum identity", flush=True)
    y = layer(xd)
    y.sum().backward()
    S = x.double().sum(0, keepdim=True).requires_grad_()
    w64 = w.double().requires_grad_()
    yS = O.layer_forward("geom", S, w64)
    yS.sum().backward()
    assert rel_err(y.detach().double().sum(0, keepdim=True), yS) <= TOL
    assert rel_err(layer.weight.grad, w64.grad) <= TOL
    x1 = x[:1].double().requires_grad_()
    O.layer_forward("geom", x1, w.double()).sum().backward()
    assert rel_err(xd.grad, x1.grad.expand(B, 256)) <= TOL


@pytest.mark.parametrize("metric", [(1,) * 8, (1, -1) * 4], ids=["++++++++", "+-+-+-+-"])
@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("batch", [1, 77, 4099])
def test_matrix_path_layer_sides(metric, side, batch):
    """Real-type n = 8: the broadcast geometric product with the weight on
    either side (matrix-representation layer kernels) against the oracle,
    values and both gradients; odd batches exercise the clamped last rows
    (which must not enter the weight gradient twice)."""
    g = torch.Generator().manual_seed(7 + side)
    x = torch.randn(batch, 256, generator=g)
    w = torch.randn(1, 256, generator=g)
    gy = torch.randn(batch, 256, generator=g)
    xd = x.cuda().requires_grad_()
    wd = w.cuda().requires_grad_()
    y = bcast.bcast_product("geom", xd, wd, metric, side=side)
    y.backward(gy.cuda())
    x64 = x.double().requires_grad_()
    w64 = w.double().requires_grad_()
    wb = w64.expand_as(x64)
    y64 = O.einsum_product("geom", x64, wb, metric) if side == 0 else O.einsum_product("geom", wb, x64, metric)
    y64.backward(gy.double())
    assert rel_err(y, y64) <= TOL
    assert rel_err(xd.grad, x64.grad) <= TOL
    assert rel_err(wd.grad, w64.grad) <= TOL


def test_layer_small_batches():
    cl = cc.CliffordAlgebra([1] * 8, device="cuda")
    layer = cc.GeometricProductLayer(cl)
    for B in (0, 1, 127, 129):
        x = torch.randn(B, 256, device="cuda", requires_grad=True)
        y = layer(x)
        y.sum().backward()
        if B:
            ref = O.layer_forward("geom", x.detach().double().cpu(), layer.weight.detach().double().cpu())
            assert rel_err(y, ref) <= TOL
        layer.weight.grad = None


@pytest.mark.parametrize("op,metric,rows", [
    ("geom", (1,) * 7, 1), ("inner", (1,) * 7, 63489), ("regressive", (1,) * 7, 17), ("lc", (-1,) * 4 + (1, 1, 0), 33),
    ("geom", (1,) * 7 + (-1,), 31745), ("wedge", (1,) * 8, 2049), ("inner", (1,) * 5 + (0, -1, 1), 300),
    ("geom", (1,) * 9, 9), ("geom", (1,) * 8 + (-1,), 15873), ("inner", (1,) * 9, 15872), ("rc", (1,) * 9, 5),
    ("geom", (1,) * 9 + (0,), 65), ("geom", (1,) * 8 + (-1, 1), 7936), ("lc", (1,) * 9 + (0,), 7937),
    ("wedge", (-1,) * 10, 3)])
@pytest.mark.parametrize("side", [0, 1])
def test_rows_path_edges(op, metric, rows, side):
    """The layers on the per-row kernels, at remainders of their row groups and
    one row below, at and above a chunk of weight gradients (31 MiB of rows):
    values and input gradient equal the per-row product's on the expanded
    weight, the weight gradient its fp64 column sums; one gradient at a time
    gives the same as both. TOL is normwise: sums of at most 1024 terms a row
    and 32 x 2 rows a partial stay below 1e-6."""
    D = 1 << len(metric)
    g = torch.Generator(device="cuda").manual_seed(rows + side)
    x, gy = (torch.randn(rows, D, device="cuda", generator=g) for _ in range(2))
    w = torch.randn(1, D, device="cuda", generator=g)
    print(f"[case] rows path op={op} metric={metric} rows={rows} side={side}", flush=True)
    x1, w1 = x.clone().requires_grad_(), w.clone().requires_grad_()
    y = bcast.bcast_product(op, x1, w1, metric, side=side)
    gx, gw = torch.autograd.grad(y, (x1, w1), gy)
    x2, w2 = x.clone().requires_grad_(), w.expand(rows, D).contiguous().requires_grad_()
    fn = {"geom": cc.geom_prod, "wedge": cc.wedge_prod, "inner": cc.inner_prod, "lc": cc.left_contraction,
          "rc": cc.right_contraction, "regressive": cc.regressive_prod}[op]
    y2 = fn(x2, w2, metric) if side == 0 else fn(w2, x2, metric)
    gx2, gw2 = torch.autograd.grad(y2, (x2, w2), gy)
    assert rel_err(y, y2) <= TOL
    assert rel_err(gx, gx2) <= TOL
    assert rel_err(gw, gw2.double().sum(0, keepdim=True)) <= TOL
    y3 = bcast.bcast_product(op, x, w1, metric, side=side)
    assert torch.equal(torch.autograd.grad(y3, w1, gy)[0], gw)
    y4 = bcast.bcast_product(op, x1, w, metric, side=side)
    assert rel_err(torch.autograd.grad(y4, x1, gy)[0], gx) <= TOL
    g0 = torch.autograd.grad(bcast.bcast_product(op, x1, w1, metric, side=side).sum(), (x1, w1))
    r0 = torch.autograd.grad(fn(x2, w2, metric).sum() if side == 0 else fn(w2, x2, metric).sum(), (x2, w2))
    assert rel_err(g0[0], r0[0]) <= TOL
    assert rel_err(g0[1], r0[1].double().sum(0, keepdim=True)) <= TOL


@pytest.mark.parametrize("op,metric", [("wedge", (1,) * 8), ("geom", (1,) * 7), ("geom", (1,) * 10), ("lc", (1,) * 9)])
@pytest.mark.parametrize("at", [0, 3])
def test_weight_inside_the_output(op, metric, at):
    """The C entry points take a weight that lies in the output's memory (row
    `at` of it): the result is the one of a separate weight, forward and input
    gradient, also without a workspace of the caller's."""
    from cliffordcuda_amd import _lib
    lib, code, n, rows = _lib.load(), O.OPS.index(op), len(metric), 77
    D = 1 << n
    g = torch.Generator(device="cuda").manual_seed(n)
    x, gy, w = (torch.randn(r, D, device="cuda", generator=g) for r in (rows, rows, 1))
    x1, w1 = x.clone().requires_grad_(), w.clone().requires_grad_()
    y = bcast.bcast_product(op, x1, w1, metric)
    gx, gw = torch.autograd.grad(y, (x1, w1), gy)
    nbytes = lib.clf_product_bcast_ws_bytes(n, rows)
    ws = torch.empty(nbytes // 4, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    neg = sum(1 << k for k, m in enumerate(metric) if m < 0)

    def into(call):
        out, got_w = torch.zeros(rows, D, device="cuda"), torch.empty(1, D, device="cuda")
        out[at] = w[0]
        torch.cuda.synchronize()
        _lib.check(call(out.data_ptr(), out[at].data_ptr(), got_w.data_ptr()), "bcast")
        return out, got_w

    print(f"[case] weight inside the output op={op} metric={metric} at={at}", flush=True)
    out, _ = into(lambda o, wp, _: lib.clf_product_bcast_fwd(code, 0, n, neg, 0, x.data_ptr(), wp, o, rows,
                                                             ws.data_ptr(), nbytes, stream))
    assert rel_err(out, y) <= TOL
    out, got_w = into(lambda o, wp, q: lib.clf_product_bcast_bwd(code, 0, n, neg, 0, x.data_ptr(), wp, gy.data_ptr(), o,
                                                                 q, rows, ws.data_ptr(), nbytes, stream))
    assert rel_err(out, gx) <= TOL and rel_err(got_w, gw) <= TOL
    out, got_w = into(lambda o, wp, q: lib.clf_product_bcast_bwd_noalloc(code, 0, n, neg, 0, x.data_ptr(), wp,
                                                                         gy.data_ptr(), o, q, rows, stream))
    assert rel_err(out, gx) <= TOL and rel_err(got_w, gw) <= TOL
