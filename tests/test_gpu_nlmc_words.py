"""The streaming mesher on sign words: chunk borders off the 64-point words, the
smallest grids, and spacings on either side of the one from which no triangle
can be degenerate (1e-4; below it the filter runs).

The map's device and host values differ by some 1e-14. A vertex differs only if
that decides a midpoint's sign or its |value| < 1e-8 stop; over the spacings
used the values are spread over 1e-5 and more, so that is expected for fewer
than one vertex in 1e6: vertices must agree to 1e-12, triangles exactly."""
import numpy as np
import pytest

import oracle as O
from quijibo_amd import api, workloads as W
from quijibo_amd._lib import FP32_BAND, FP64, MAP_BLACK_HOLE

pytestmark = pytest.mark.gpu


def polys(w):
    return O.poly(w.top.roots, w.top.powers), O.poly(w.bottom.roots, w.bottom.powers)


def surface_point(w):
    """A point with F = 0 between two grid points of opposite sign."""
    res = (24, 24, 24)
    p = O.make_params(w.max_iter, 2000.0, w.exp_scaling, w.slice, O.BLACK_HOLE)
    f = O.field_map(O.make_grid(res, w.center, w.lengths), *polys(w), p).reshape(24, 24, 24)
    z, y, x = np.argwhere((f[:, :, :-1] > 0) != (f[:, :, 1:] > 0))[17]
    at = lambda i: np.array([w.center[k] - w.lengths[k] / 2 + w.lengths[k] / 24 * (i[k] + 0.5) for k in range(3)])
    a, b = at((x, y, z)), at((x + 1, y, z))
    value = lambda q: O.points_eval(q, *polys(w), p)[0]
    sign = value(a) > 0
    for _ in range(40):
        m = (a + b) / 2
        if (value(m) > 0) == sign:
            a = m
        else:
            b = m
    return tuple(a)


@pytest.mark.parametrize("spacing", [4e-6, 0.9e-4, 1.1e-4])
@pytest.mark.parametrize("res,chunk", [((2, 2, 2), 64), ((3, 2, 65), 7), ((9, 7, 11), 1), ((17, 31, 12), 5),
                                       ((33, 8, 20), 64)])
def test_nonlinear_words_match_the_oracle(gpu, res, chunk, spacing):
    w = W.config2(8)
    center = surface_point(w)
    lengths = tuple(spacing * r for r in res)
    ov, ot, bad = O.nonlinear_mc(O.make_grid(res, center, lengths), *polys(w),
                                 O.make_params(w.max_iter, 2000.0, w.exp_scaling, w.slice, O.BLACK_HOLE), 0.0)
    assert bad == 0 and len(ot) > 0
    g = api.make_grid(res, center, lengths)
    r = api.Rational(api.POLYNOMIAL_4D(w.top.roots, w.top.powers), api.POLYNOMIAL_4D(w.bottom.roots, w.bottom.powers))
    p = api.make_params(w.max_iter, 2000.0, w.exp_scaling, w.slice, MAP_BLACK_HOLE)
    for precision in (FP64, FP32_BAND):
        v, t = api.nonlinear_mesh(g, r, p, 0.0, precision, 0.05, chunk, workspace=api.Workspace())
        print(res, chunk, spacing, len(v), len(t), len(ov), len(ot), flush=True)
        assert np.array_equal(t, ot)
        assert v.shape == ov.shape and np.abs(v - ov).max() <= 1e-12
