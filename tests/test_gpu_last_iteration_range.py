"""The last iteration's norms at the ends of FP64's range: 60 to 120 roots close
to the centre with exponents 3 to 4.2, so that over the grid |T|^2, |B|^2 and
|q|^2 pass 2^-1022, 2^-950, 1, 2^950 and 2^1023, where norms and products meet.

Tolerance 1e-8 max(1, |F|) as for other sets of up to 256 roots, and the same
non-finite cells. Where |q|^2 is below 2^-1010 (F < -350) its denormal rounding
decides the value and whether it is 0, so there F only has to be that small."""
import numpy as np
import pytest

import oracle as O
from quijibo_amd import api
from quijibo_amd._lib import FP64, FP64_EXACT, MAP_BLACK_HOLE

pytestmark = pytest.mark.gpu

RES, LENGTHS = (14, 13, 12), (3.2, 3.0, 2.8)


@pytest.mark.parametrize("nt, nb, kind", [(120, 0, "real"), (120, 60, "real"), (60, 120, "real"), (110, 110, "real"),
                                          (120, 60, "mixed"), (60, 120, "mixed"), (120, 0, "mixed")])
@pytest.mark.parametrize("scaling", [1.0, 1e-80, 1e80])
def test_norms_and_products_meet(gpu, nt, nb, kind, scaling):
    rng = np.random.default_rng(nt + 3 * nb)
    roots = [rng.normal(scale=0.05, size=(n, 4)) for n in (nt, nb)]
    powers = [rng.uniform(3.0, 4.2, size=n) for n in (nt, nb)]
    if kind == "mixed":
        for p in powers:
            p[::3], p[1::3] = 1.0, 2.0
            p[2::3] = 4.2
    g = O.make_grid(RES, (0.0, 0.0, 0.0), LENGTHS)
    ref = O.field_map(g, O.poly(roots[0], powers[0], 1.0), O.poly(roots[1], powers[1], 1.0),
                      O.make_params(1, 2000.0, scaling, 0.0, O.BLACK_HOLE))
    r = api.Rational(api.POLYNOMIAL_4D(roots[0], powers[0], 1.0), api.POLYNOMIAL_4D(roots[1], powers[1], 1.0))
    p = api.make_params(1, 2000.0, scaling, 0.0, MAP_BLACK_HOLE)
    for prec in (FP64, FP64_EXACT):
        F = api.field_eval(api.make_grid(RES, (0.0, 0.0, 0.0), LENGTHS), r, p, prec).cpu().numpy()
        low = ref < -350.0
        assert np.all(F[low] < -349.0)
        assert np.array_equal(np.isfinite(F[~low]), np.isfinite(ref[~low]))
        m = ~low & np.isfinite(ref)
        e = np.abs(F[m] - ref[m]) / np.maximum(1.0, np.abs(ref[m]))
        print("%d+%d %s: %.1e over %d, %d low, %d not finite, F %.0f to %.0f" % (
            nt, nb, kind, e.max(), m.sum(), low.sum(), (~np.isfinite(ref)).sum(), ref[m].min(), ref[m].max()))
        assert e.max() <= 1e-8
