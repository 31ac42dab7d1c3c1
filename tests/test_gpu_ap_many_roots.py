"""The AP pass where a wave's roots are more than it keeps logarithms of (129 roots
and more on grids of 256-cell blocks): cells with a gradient listed over many
blocks, blocks without any (the origin's, saturated ones), ragged ends. Against
the oracle, tolerance 1e-9 relative, the AP pass's own (tests/test_gpu_grad.py)."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api
from quijibo_amd._lib import MAP_ADAPTIVE, MAP_SKIP_ORIGIN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res, nt, nb, alpha", [((33, 32, 32), 64, 64, 2.0), ((33, 32, 32), 70, 66, 2.0),
                                                ((35, 31, 33), 70, 66, 300.0), ((32, 32, 32), 130, 131, 2.0)])
def test_recomputed_logarithms(gpu, res, nt, nb, alpha):
    rng = np.random.default_rng(nt)
    tr, br = rng.normal(scale=0.6, size=(nt, 4)), rng.normal(scale=0.6, size=(nb, 4))
    tr[:, 3] *= 0.1
    br[:, 3] *= 0.1
    tp, bp = rng.uniform(0.1, 0.5, size=nt), rng.uniform(0.1, 0.5, size=nb)
    weight = rng.normal(size=6 * 7 * 8)
    lengths = (3.0, 2.5, 2.75)
    got = api.ap_score_gradients(
        api.make_grid(res, lengths=lengths), api.Rational(api.POLYNOMIAL_4D(tr, tp, 1.1), api.POLYNOMIAL_4D(br, bp, 0.9)),
        api.make_params(1, 20.0, 0.8, 0.0, MAP_SKIP_ORIGIN | MAP_ADAPTIVE), api.make_grid((6, 7, 8), lengths=lengths),
        torch.from_numpy(weight).cuda(), alpha, 0.1)
    ref = O.ap_score_gradients(
        O.make_grid(res, (0.0, 0.0, 0.0), lengths), O.poly(tr, tp, 1.1), O.poly(br, bp, 0.9),
        O.make_params(1, 20.0, 0.8, 0.0, O.SKIP_ORIGIN | O.AP_REPASS),
        O.make_grid((6, 7, 8), (0.0, 0.0, 0.0), lengths), weight, alpha, 0.1)
    assert got["adaptive_cells"] == ref["overflowed"]
    for k in ("score", "grad_exp", "grad_top", "grad_bottom", "grad_top_scalar", "grad_bottom_scalar"):
        a, b = np.atleast_1d(got[k]), np.atleast_1d(ref[k])
        assert np.max(np.abs(a - b)) <= 1e-9 * np.max(np.abs(b)), k
    assert np.allclose(got["field"].cpu().numpy(), ref["field"], rtol=1e-9, atol=1e-12)
