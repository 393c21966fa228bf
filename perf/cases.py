"""What the performance of this framework is judged by: calls that a program
using it makes, through its public entry points, from single-row latencies to
batches that fill the card.

A case is a dict of plain values:
  kind    "product"  CliffordAlgebra product methods (and graded ops) on rows
          "layer"    a product layer's training step (weight shared by the batch)
          "rotor"    RotorLayer's training step, or apply_rotor with a kept rotor
  metric  the signature, one character per generator: "+", "-" or "0"
  ops     comma-separated ops of a "product" case, run one after the other
  grad    True: forward and backward; False: forward only
  batch   rows

Everything is fp32, as the framework is.
"""
import math

import torch

import cliffordcuda_amd as cc

DEVICE = "cuda"

METHODS = {"geom": "geom_prod", "wedge": "wedge_prod", "inner": "inner_prod", "lc": "left_contraction",
           "rc": "right_contraction", "regressive": "regressive_prod"}
LAYERS = {"geom": "GeometricProductLayer", "wedge": "WedgeProductLayer", "inner": "InnerProductLayer",
          "lc": "LeftContractionLayer", "rc": "RightContractionLayer", "regressive": "RegressiveProductLayer"}
MASKED = ("wedge", "inner", "lc", "rc", "regressive")


def listed():
    return [
        # The smallest ordinary call: one forward product of a small algebra on
        # a thousand rows, where the launch is most of the time.
        {"name": "geom_n5_forward", "kind": "product", "metric": "+++++", "ops": "geom", "grad": False,
         "batch": 1024},
        # The headline workload: Cl(8,0) geometric product, forward and
        # backward, on a batch that fills the card (2 GB of rows).
        {"name": "geom_n8_large", "kind": "product", "metric": "++++++++", "ops": "geom", "grad": True,
         "batch": 262144},
        # The other five products of a Cl(6,1) model, forward and backward.
        {"name": "masked_n7", "kind": "product", "metric": "++++++-", "ops": "wedge,inner,lc,rc,regressive",
         "grad": True, "batch": 65536},
        # A degenerate (projective) algebra: products forward and backward,
        # with the norm and a grade projection that such a model also takes.
        {"name": "degenerate_n10", "kind": "product", "metric": "+++++++++0", "ops": "geom,lc,norm_sq,project2",
         "grad": True, "batch": 16384},
        # A spacetime-like signature at n = 8 (not a real matrix algebra), on
        # an odd number of rows.
        {"name": "geom_n8_cl71", "kind": "product", "metric": "+++++++-", "ops": "geom", "grad": True,
         "batch": 50001},
        # A small algebra whose generators come in the user's own order, with a
        # null one among them: the general signature path.
        {"name": "mixed_n6", "kind": "product", "metric": "++++0-", "ops": "geom,inner,lc", "grad": True,
         "batch": 30011},
        # The largest algebra of the published latency table at its largest
        # batch: a few rows of 4096 coefficients.
        {"name": "geom_n12_few_rows", "kind": "product", "metric": "++++++++++++", "ops": "geom", "grad": True,
         "batch": 64},
        # The same kind of algebra on a training batch of odd size.
        {"name": "geom_n11_rows", "kind": "product", "metric": "++++++++++-", "ops": "geom", "grad": True,
         "batch": 1999},
        # The geometric product layer's training step at a large batch.
        {"name": "layer_geom_n8", "kind": "layer", "metric": "++++++++", "ops": "geom", "grad": True,
         "batch": 262144},
        # Another product's layer, at a batch that is not a multiple of any tile.
        {"name": "layer_inner_n8", "kind": "layer", "metric": "++++++++", "ops": "inner", "grad": True,
         "batch": 60013},
        # RotorLayer's training step: compile, sandwich, both gradients.
        {"name": "rotor_n8_train", "kind": "rotor", "metric": "+++++++-", "ops": "rotor", "grad": True,
         "batch": 131072},
        # A kept rotor applied to a few rows, as the published table times it.
        {"name": "rotor_n11_apply", "kind": "rotor", "metric": "+++++++++++", "ops": "rotor", "grad": False,
         "batch": 64},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    """One more case of the listed ones' ranges. Batches are log-uniform; the
    cap keeps rows * 4^n (the terms of a geometric product) and the rows' bytes
    below those of the largest listed cases."""
    family = rng.choice(["euclid", "signature", "mixed", "degenerate", "layer", "rotor"])
    if family == "euclid":  # the published table's algebras, from one row upwards
        n = rng.randint(7, 12)
        ops, grad, low, high = rng.choice(("geom",) + MASKED), rng.random() < 0.6, 1, 60000
        metric = "+" * n
    elif family == "signature":  # Cl(p, q), the usual order
        n = rng.randint(4, 11)
        q = rng.randint(1, min(4, n - 1))
        ops, grad, low, high = rng.choice(("geom", "geom") + MASKED), rng.random() < 0.8, 256, 200000
        metric = "+" * (n - q) + "-" * q
    elif family == "mixed":  # any order of +, - and 0
        n = rng.randint(4, 7)
        ops, grad, low, high = rng.choice(("geom", "inner", "lc", "rc", "wedge")), rng.random() < 0.8, 256, 60000
        metric = "".join(rng.choice("++--0") for _ in range(n))
    elif family == "degenerate":  # one null generator, last
        n = rng.randint(8, 10)
        ops, grad, low, high = rng.choice(("geom", "lc", "rc", "inner", "geom,norm_sq,project2")), True, 64, 16384
        metric = "+" * (n - 1) + "0"
    elif family == "layer":
        n = rng.randint(7, 10)
        q = rng.randint(0, 1)
        ops, grad, low, high = rng.choice(("geom", "geom") + MASKED), True, 256, 262144
        metric = "+" * (n - q) + "-" * q
    else:
        n = rng.randint(7, 12)
        ops, grad, low, high = "rotor", rng.random() < 0.6, 1, 131072
        metric = "+" * n
    terms = {"mixed": 4 ** 6 * 60000, "layer": 4 ** 8 * 65536}.get(family, 4 ** 11 * 1999)
    if family != "rotor":
        high = min(high, terms // 4 ** n)
    high = min(high, (1 << (25 if family == "rotor" else 26)) >> n)
    kind = family if family in ("layer", "rotor") else "product"
    return {"kind": kind, "metric": metric, "ops": ops, "grad": grad,
            "batch": _log_int(rng, low, max(low, high))}


def _signature(case):
    return [{"+": 1, "-": -1, "0": 0}[c] for c in case["metric"]]


def _inputs(case, seed):
    """Coefficients, weights and upstream gradients ~ N(0, 1), the layers' own
    initialisation included; the same values for prepare and exact."""
    n = len(case["metric"])
    dim, batch = 1 << n, case["batch"]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=DEVICE)

    if case["kind"] == "product":
        names = ("a", "b", "g") if case["grad"] else ("a", "b")
        return {k: normal(batch, dim) for k in names}
    rows = {"x": normal(batch, dim)}
    if case["grad"]:
        rows["g"] = normal(batch, dim)
    rows["w"] = normal(1, dim if case["kind"] == "layer" else n * (n - 1) // 2)
    return rows


def prepare(case, seed):
    state = dict(_inputs(case, seed))
    cl = cc.CliffordAlgebra(_signature(case), device=DEVICE)
    state.update(cl=cl, kind=case["kind"], ops=case["ops"].split(","), grad=case["grad"])
    if case["kind"] == "product":
        state["a0"] = state["a"].detach()
        for k in ("a", "b"):
            state[k].requires_grad_(case["grad"])
    elif case["kind"] == "layer":
        state["layer"] = getattr(cc, LAYERS[case["ops"]])(cl)
        with torch.no_grad():
            state["layer"].weight.copy_(state["w"])
        state["x"].requires_grad_()
    elif case["grad"]:
        state["layer"] = cc.RotorLayer(cl)
        with torch.no_grad():
            state["layer"].bivector.copy_(state["w"])
        state["x"].requires_grad_()
    else:
        state["cs"] = cl.compile_bivector(state["w"])
    return state


def run(state):
    if state["kind"] == "product":
        cl, a, b = state["cl"], state["a"], state["b"]
        out = []
        for op in state["ops"]:
            if op == "norm_sq":
                out.append(cl.norm_sq(state["a0"]))
            elif op == "project2":
                out.append(cl.grade_projection(state["a0"], 2))
            elif state["grad"]:
                c = getattr(cl, METHODS[op])(a, b)
                out += [c, *torch.autograd.grad(c, (a, b), state["g"])]
            else:
                out.append(getattr(cl, METHODS[op])(a, b))
        return out
    if "layer" in state:
        layer, x = state["layer"], state["x"]
        y = layer(x)
        return [y, *torch.autograd.grad(y, (x, *layer.parameters()), state["g"])]
    return [state["cl"].apply_rotor(state["cs"], state["x"])]


def work(case):
    """Bytes: the pass's inputs once, its outputs once. Operations: a geometric
    product as one product of matrices of side 2^ceil(n / 2) and (n odd) half
    as many terms, the masked products by their nonzero terms, a rotor as two
    products; a backward is twice its forward."""
    n, batch = len(case["metric"]), case["batch"]
    row = 4 * (1 << n)
    nul = case["metric"].count("0")
    passes = 3 if case["grad"] else 1
    matrix = 2 * (1 << n) * (1 << ((n + 1) // 2))
    one_sided = 3 ** (n - nul) * 2 ** nul
    flops = {"geom": matrix, "wedge": 2 * 3 ** n, "regressive": 2 * 3 ** n, "lc": 2 * one_sided, "rc": 2 * one_sided,
             "inner": 2 * (2 * one_sided - 2 ** (n - nul)), "rotor": 2 * matrix}
    ops = case["ops"].split(",")
    total_flops, out_rows, out_bytes = 0, 0, 0
    for op in ops:
        if op == "norm_sq":
            total_flops += 2 * (1 << n)
            out_bytes += 4 * batch
        elif op == "project2":
            out_rows += 1
        else:
            total_flops += passes * flops[op]
            out_rows += (3 if case["kind"] == "product" else 2) if case["grad"] else 1
    in_rows = (3 if case["grad"] else 2) if case["kind"] == "product" else (2 if case["grad"] else 1)
    return {"bytes": (in_rows + out_rows) * row * batch + out_bytes, "flops": total_flops * batch}


def tolerance(case):
    """fp32 sums of up to 4096 signed terms per coefficient, in any order or
    factorisation, a rotor's chain of planes, and a parameter gradient's sum
    over the batch: four times the largest error measured against exact()."""
    return {"rel": 4e-6}


# ---- the same in 64 bits ---------------------------------------------------

def _sign_table(op, metric):
    """s[i, j] of e_i e_j = s e_{i^j} for the terms that op keeps."""
    n = len(metric)
    k = torch.arange(1 << n, device=DEVICE)
    popc = sum((k >> b) & 1 for b in range(n))
    i, j = k.view(-1, 1), k.view(1, -1)
    swaps = sum(((j >> b) & 1) * popc[i >> (b + 1)] for b in range(n))
    s = (1 - 2 * (swaps & 1)).to(torch.float64)
    if op == "wedge":
        return s * ((i & j) == 0)
    for b, m in enumerate(metric):
        if m != 1:
            s = torch.where(((i & j) >> b) & 1 == 1, s * m, s)
    keep = {"geom": None, "lc": (i & ~j) == 0, "rc": (j & ~i) == 0,
            "inner": ((i & ~j) == 0) | ((j & ~i) == 0)}[op]
    return s if keep is None else s * keep


def _xor_sum(x, y, weight):
    """out[:, k] = sum_i weight[i, k] x[:, i] y[:, i ^ k]."""
    out = torch.zeros_like(y)
    k = torch.arange(y.shape[1], device=y.device)
    for i in range(x.shape[1]):
        out.addcmul_(x[:, i:i + 1], y[:, k ^ i] * weight[i])
    return out


def _product64(op, metric, a, b, g):
    """[c], or [c, ga, gb] when an upstream gradient is given."""
    dim = a.shape[1]
    if op == "regressive":  # dual(dual a ^ dual b), dual(x) = x I^-1
        full = dim - 1
        s = _sign_table("geom", metric)
        sign = s[:, full] / s[full, full]  # x_j e_j -> sign[j] e_{~j}

        def dual(x):
            return (x * sign).flip(1)

        def dual_adjoint(x):
            return x.flip(1) * sign

        out = _product64("wedge", metric, dual(a), dual(b), None if g is None else dual_adjoint(g))
        return [dual(out[0])] + [dual_adjoint(t) for t in out[1:]]
    s = _sign_table(op, metric)
    k = torch.arange(dim, device=a.device)
    xor = k.view(-1, 1) ^ k.view(1, -1)
    out = [_xor_sum(a, b, s.gather(1, xor))]
    if g is not None:
        # ga[m] = sum_k s[m, m^k] g[k] b[m^k], gb[m] = sum_k s[m^k, m] g[k] a[m^k]
        out.append(_xor_sum(g, b, s.gather(1, xor).t().contiguous()))
        out.append(_xor_sum(g, a, s.gather(0, xor)))
    return out


def _layer64(op, metric, x, w, g):
    """y = x M with M[i, k] = s[i, i^k] w[i^k]; the regressive layer's M from
    the products of the unit blades."""
    dim = x.shape[1]
    if op == "regressive":
        eye = torch.eye(dim, dtype=torch.float64, device=x.device)
        m = _product64(op, metric, eye, w.expand(dim, dim).contiguous(), None)[0]
        y, gx = x @ m, g @ m.t()
        # gw = sum over rows of the product's gradient to w, through G = x^T g
        big = x.t() @ g
        gw = _product64(op, metric, eye, eye, big)[2].sum(0, keepdim=True)
        return [y, gx, gw]
    s = _sign_table(op, metric)
    k = torch.arange(dim, device=x.device)
    xor = k.view(-1, 1) ^ k.view(1, -1)
    sig = s.gather(1, xor)
    m = sig * w.view(-1)[xor]
    big = (x.t() @ g) * sig
    gw = torch.zeros(dim, dtype=torch.float64, device=x.device).scatter_add_(0, xor.reshape(-1), big.reshape(-1))
    return [x @ m, g @ m.t(), gw.view(1, -1)]


def _rotor64(n, x, biv, g):
    """~R x R with R = exp(B), B = sum b_m e_i e_j: the exponential of the map
    x -> x B - B x on the coefficients."""
    dim = 1 << n
    s = _sign_table("geom", [1] * n)
    k = torch.arange(dim, device=x.device)
    planes = [(1 << i) | (1 << j) for i in range(n) for j in range(i + 1, n)]
    biv = biv.view(-1).detach().requires_grad_(g is not None)
    gen = torch.zeros(dim, dim, dtype=torch.float64, device=x.device)
    for m, p in enumerate(planes):
        coef = (s[k, p] - s[p, k])
        step = torch.zeros_like(gen)
        step[k ^ p, k] = coef
        gen = gen + biv[m] * step
    rot = torch.linalg.matrix_exp(gen)
    y = x @ rot.t()
    if g is None:
        return [y.detach()]
    gb, = torch.autograd.grad(rot, (biv,), g.t() @ x)
    return [y.detach(), g @ rot.detach(), gb.view(1, -1)]


def exact(case, seed):
    n = len(case["metric"])
    if case["kind"] == "rotor" and n == 12 and case["grad"]:
        return None  # the exponential's derivative over 4096 x 4096 takes too long
    metric = _signature(case)
    v = {k: t.double() for k, t in _inputs(case, seed).items()}
    if case["kind"] == "rotor":
        return _rotor64(n, v["x"], v["w"], v.get("g"))
    if case["kind"] == "layer":
        return _layer64(case["ops"], metric, v["x"], v["w"], v["g"])
    out = []
    for op in case["ops"].split(","):
        if op == "norm_sq":
            weight = torch.ones(1 << n, dtype=torch.float64, device=DEVICE)
            k = torch.arange(1 << n, device=DEVICE)
            for b, m in enumerate(metric):
                weight = torch.where((k >> b) & 1 == 1, weight * m, weight)
            out.append((v["a"] ** 2) @ weight)
        elif op == "project2":
            k = torch.arange(1 << n, device=DEVICE)
            out.append(v["a"] * (sum((k >> b) & 1 for b in range(n)) == 2))
        else:
            out += _product64(op, metric, v["a"], v["b"], v.get("g"))
    return out
