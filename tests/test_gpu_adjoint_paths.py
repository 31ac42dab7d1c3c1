"""The adjoint where its branches meet, against torch autograd of the map in
float64 on the CPU: 4 to 32 lanes per point with ragged shares, exponents 1, 2
and real, more iterations than the kept products, points that escape early,
points without a gradient, no bottom roots.

Tolerances relative to the gradient's norm: FP64 1e-8 (rounding 1e-15 per
product, amplified by at most about 30 per iteration), FP32 2e-3, the gradient
tests' own (tests/test_gpu_grad.py)."""
import math

import numpy as np
import pytest
import torch

from quijibo_amd import api
from quijibo_amd._lib import FP32_BAND, FP64, MAP_BLACK_HOLE

pytestmark = pytest.mark.gpu


def _mul(a, b):
    return (a[0] * b[0] - a[1] * b[1] - a[2] * b[2] - a[3] * b[3], a[0] * b[1] + a[1] * b[0] + a[2] * b[3] - a[3] * b[2],
            a[0] * b[2] - a[1] * b[3] + a[2] * b[0] + a[3] * b[1], a[0] * b[3] + a[1] * b[2] - a[2] * b[1] + a[3] * b[0])


def _product(q, roots, powers):
    unit, ln = None, 0.0
    for i in range(roots.shape[0]):
        b = tuple(q[k] - roots[i, k] for k in range(4))
        v = (b[1] ** 2 + b[2] ** 2 + b[3] ** 2).sqrt()
        m = powers[i] * torch.atan2(v, b[0])
        f = torch.sin(m) / v
        u = (torch.cos(m), f * b[1], f * b[2], f * b[3])
        ln = ln + powers[i] * torch.log((b[0] ** 2 + v ** 2).sqrt())
        unit = u if unit is None else _mul(unit, u)
    return unit, ln


def _reference(pts, tr, tp, br, bp, g, iters, c, escape):
    leaves = [torch.from_numpy(x).requires_grad_() for x in (tr, tp, br, bp)]
    q = tuple(torch.from_numpy(pts[:, k].copy()) for k in range(3)) + (torch.zeros(len(pts), dtype=torch.float64),)
    F = torch.log(sum(x * x for x in q).sqrt())
    live = F < math.log(escape)
    for _ in range(iters):
        q = tuple(torch.where(live, x, torch.full_like(x, 0.3)) for x in q)
        unit, ln = _product(q, leaves[0], leaves[1])
        if len(br):
            ub, lb = _product(q, leaves[2], leaves[3])
            unit, ln = _mul(unit, (ub[0], -ub[1], -ub[2], -ub[3])), ln - lb
        ln = ln + math.log(c)
        F = torch.where(live, ln, F)
        live = live & (F < math.log(escape))
        s = torch.where(live, ln, torch.zeros_like(ln)).exp()
        q = tuple(x * s for x in unit)
    (F * torch.from_numpy(g)).sum().backward()
    gr = [x.grad if x.grad is not None else torch.zeros_like(x) for x in leaves]
    return (torch.cat([gr[0].reshape(-1, 4), gr[2].reshape(-1, 4)]).numpy(),
            torch.cat([gr[1].reshape(-1), gr[3].reshape(-1)]).numpy())


@pytest.mark.parametrize("n, nt, nb, powers, iters", [
    (1, 1, 0, "ones", 1),       # one point, one root
    (5, 3, 2, "real", 2),       # 8 lanes, most of them without a root
    (70, 13, 12, "int", 3),     # 16 lanes, one root a lane
    (33, 40, 9, "ones", 2),     # 32 lanes, uneven polynomials
    (130, 6, 6, "ones", 5),     # more iterations than kept products
    (8200, 5, 4, "real", 2),    # 4 lanes
    (8200, 17, 3, "int", 1),    # 8 lanes, one iteration
    (8200, 33, 32, "ones", 2),  # 16 lanes
    (9, 410, 409, "ones", 1),   # the most roots: 96 KiB of LDS
])
def test_adjoint_against_autograd(gpu, n, nt, nb, powers, iters):
    rng = np.random.default_rng(7 * n + nt)
    tr, br = rng.normal(scale=0.6, size=(nt, 4)), rng.normal(scale=0.6, size=(nb, 4))
    make = {"ones": lambda m: np.ones(m), "int": lambda m: rng.integers(1, 3, size=m).astype(float),
            "real": lambda m: rng.uniform(0.5, 1.8, size=m)}[powers]
    tp, bp = make(nt), make(nb)
    pts = rng.uniform(-1.0, 1.0, size=(n, 3))
    pts[::7] *= 6.0  # some escape early (escape radius 20)
    g = rng.normal(size=n)
    g[3::11] = 0.0
    gr, gp = _reference(pts, tr, tp, br, bp, g, iters, 0.8, 20.0)
    r = api.Rational(api.POLYNOMIAL_4D(tr, tp), api.POLYNOMIAL_4D(br, bp))
    p = api.make_params(iters, 20.0, 0.8, 0.0, MAP_BLACK_HOLE)
    for prec, tol in ((FP64, 1e-8), (FP32_BAND, 2e-3)):
        a, b = api.points_adjoint(torch.from_numpy(pts).cuda(), r, p, torch.from_numpy(g).cuda(), prec)
        ea = np.linalg.norm(a.cpu().numpy() - gr) / np.linalg.norm(gr)
        eb = np.linalg.norm(b.cpu().numpy() - gp) / np.linalg.norm(gp)
        print("%d points %d+%d %s x%d prec %d: %.2e %.2e" % (n, nt, nb, powers, iters, prec, ea, eb), flush=True)
        assert ea <= tol and eb <= tol
