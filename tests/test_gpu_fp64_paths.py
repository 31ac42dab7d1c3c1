"""The FP64 evaluators where their branches meet, against the oracle: the last
iteration from magnitudes (groups of 8 roots and their remainders, products
beyond FP64's range, which take the full product), polar powers (exponents 0,
below 1, negative, large; bases on the real axis and on a root) and the
extended range with the exponent taken out per group.

Tolerance 1e-9 max(1, |F|) and the same non-finite cells, the field tests' own
(tests/test_gpu_field.py, tests/test_gpu_extended.py)."""
import numpy as np
import pytest

import oracle as O
from quijibo_amd import api, workloads as W
from quijibo_amd._lib import FP64, FP64_EXACT, MAP_BLACK_HOLE, MAP_EXTENDED_RANGE

pytestmark = pytest.mark.gpu

RES, LENGTHS = (10, 9, 7), (3.0, 2.7, 2.1)


def _roots(rng, n):
    return np.concatenate([rng.normal(scale=0.6, size=(n, 3)), rng.uniform(-0.1, 0.1, size=(n, 1))], axis=1)


def _workload(nt, nb, kind, iters):
    rng = np.random.default_rng(100 * nt + nb + iters)
    tr, br = _roots(rng, nt), _roots(rng, nb)
    tp, bp = rng.integers(1, 3, size=nt).astype(float), rng.integers(1, 3, size=nb).astype(float)
    if kind != "int":
        tp, bp = rng.uniform(0.3, 1.8, size=nt), rng.uniform(0.3, 1.8, size=nb)
        tp[0] = 1.0
    if kind == "mixed":
        tp[1], bp[0], bp[1] = 0.0, 2.0, -0.6
    if kind == "axis":  # cell centres on the line through root 0 and on root 1
        c = [-LENGTHS[i] / 2 + (np.array([4, 3, 3])[i] + 0.5) * LENGTHS[i] / RES[i] for i in range(3)]
        tr[0] = [c[0] + 0.11, c[1], c[2], 0.0]
        tr[1] = [c[0], c[1], c[2], 0.0]
        tp[0] = 0.7
    if kind == "range":  # running products pass FP64's range in parts of the grid
        tp[0], bp[0] = 900.0, 880.0
    return W.Workload("fp64", RES, W.RootSet(tr, tp), W.RootSet(br, bp), max_iter=iters, lengths=LENGTHS)


@pytest.mark.parametrize("nt, nb, kind, iters", [
    (1, 0, "int", 1), (1, 1, "real", 2), (7, 8, "int", 2), (9, 16, "int", 3), (17, 7, "real", 2), (8, 9, "mixed", 2),
    (5, 4, "mixed", 1), (6, 3, "axis", 1), (6, 3, "axis", 2), (4, 4, "range", 1), (4, 4, "range", 2),
])
@pytest.mark.parametrize("ext", [False, True])
def test_fp64_evaluators(gpu, nt, nb, kind, iters, ext):
    w = _workload(nt, nb, kind, iters)
    p = api.make_params(w.max_iter, w.escape, 0.9, 0.0, MAP_BLACK_HOLE | (MAP_EXTENDED_RANGE if ext else 0))
    r = api.Rational(api.POLYNOMIAL_4D(w.top.roots, w.top.powers, 1.0),
                     api.POLYNOMIAL_4D(w.bottom.roots, w.bottom.powers, 1.0))
    ref = O.field_map(O.make_grid(RES, w.center, LENGTHS), O.poly(w.top.roots, w.top.powers, 1.0),
                      O.poly(w.bottom.roots, w.bottom.powers, 1.0),
                      O.make_params(w.max_iter, w.escape, 0.9, 0.0, O.BLACK_HOLE | (O.EXTENDED if ext else 0)))
    fin = np.isfinite(ref)
    for prec in (FP64, FP64_EXACT):
        F = api.field_eval(api.make_grid(RES, w.center, LENGTHS), r, p, prec).cpu().numpy()
        # an overflowed product is infinite or NaN by the order of its sums, so only the class is compared
        assert np.array_equal(np.isfinite(F), fin)
        e = np.abs(F[fin] - ref[fin]) / np.maximum(1.0, np.abs(ref[fin]))
        print("%d+%d %s x%d ext %d: %.2e, %d not finite" % (nt, nb, kind, iters, ext, e.max(), (~fin).sum()))
        assert e.max() <= 1e-9
