"""The AP pass where the sum of e |log|b|| over both polynomials is out of the fast
kernel's range in some cells and each polynomial's alone is within it (they are
taken from logarithms in the second kernel), beside cells where it is not (taken by
the formulas) and several groups of 256 cells per block.
Against the oracle, tolerance 1e-9 relative, the AP pass's own
(tests/test_gpu_grad.py)."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api
from quijibo_amd._lib import MAP_ADAPTIVE, MAP_SKIP_ORIGIN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res, n, e", [((16, 15, 14), 20, 11.0), ((17, 16, 15), 20, 17.5),
                                       ((64, 48, 49), 9, 25.0)])
def test_sum_beyond_the_range(gpu, res, n, e):
    rng = np.random.default_rng(n)
    tr, br = rng.normal(scale=0.6, size=(n, 4)), rng.normal(scale=0.6, size=(n, 4))
    tr[:, 3] *= 0.1
    br[:, 3] *= 0.1
    tp, bp = rng.uniform(0.5 * e, 1.5 * e, size=n), rng.uniform(0.5 * e, 1.5 * e, size=n)
    weight = rng.normal(size=6 * 7 * 8)
    lengths = (3.0, 2.5, 2.75)
    got = api.ap_score_gradients(
        api.make_grid(res, lengths=lengths), api.Rational(api.POLYNOMIAL_4D(tr, tp, 1.1), api.POLYNOMIAL_4D(br, bp, 0.9)),
        api.make_params(1, 20.0, 0.8, 0.0, MAP_SKIP_ORIGIN | MAP_ADAPTIVE), api.make_grid((6, 7, 8), lengths=lengths),
        torch.from_numpy(weight).cuda(), 0.02, 0.1)
    ref = O.ap_score_gradients(
        O.make_grid(res, (0.0, 0.0, 0.0), lengths), O.poly(tr, tp, 1.1), O.poly(br, bp, 0.9),
        O.make_params(1, 20.0, 0.8, 0.0, O.SKIP_ORIGIN | O.AP_REPASS),
        O.make_grid((6, 7, 8), (0.0, 0.0, 0.0), lengths), weight, 0.02, 0.1)
    x, y, z = [-0.5 * l + (np.arange(k) + 0.5) * l / k for k, l in zip(res, lengths)]
    Z, Y, X = np.meshgrid(z, y, x, indexing="ij")
    q = np.stack([X.ravel(), Y.ravel(), Z.ravel(), 0 * X.ravel()], axis=1)
    st, sb = [sum(k * abs(s) * np.abs(np.log(np.linalg.norm(q - r, axis=1))) for r, s in zip(rr, pp))
              for rr, pp, k in ((tr, tp, 1.1), (br, bp, 0.9))]
    print("in range %d, by its polynomials %d, out %d" % ((st + sb < 340).sum(), ((st + sb >= 340) & (np.maximum(st, sb) < 330)).sum(),
                                                        (np.maximum(st, sb) >= 330).sum()), flush=True)
    assert ((st + sb >= 340) & (np.maximum(st, sb) < 330)).sum() > 20
    assert got["adaptive_cells"] == ref["overflowed"]
    for k in ("score", "grad_exp", "grad_top", "grad_bottom", "grad_top_scalar", "grad_bottom_scalar"):
        a, b = np.atleast_1d(got[k]), np.atleast_1d(ref[k])
        assert np.max(np.abs(a - b)) <= 1e-9 * np.max(np.abs(b)), k
    assert np.allclose(got["field"].cpu().numpy(), ref["field"], rtol=1e-9, atol=1e-11)


@pytest.mark.parametrize("res", [(16, 15, 14), (33, 32, 34)])
def test_cells_next_to_roots(gpu, res):
    """One polynomial out of range in the cells next to a root, which the second
    kernel takes by the formulas; small exponents otherwise."""
    rng = np.random.default_rng(5)
    lengths, offsets = (3.0, 2.5, 2.75), (1e-7, 1e-9)
    tr, br = rng.normal(scale=0.6, size=(7, 4)), rng.normal(scale=0.6, size=(6, 4))
    tr[:, 3] = br[:, 3] = 0.0
    og = O.make_grid(res, (0.0, 0.0, 0.0), lengths)
    for rr, k, cell in ((tr, 2, (3, 4, 5)), (br, 1, (11, 9, 2)), (tr, 4, (11, 9, 3))):
        rr[k, :3] = np.asarray(O.cell_center(og, *cell)) + np.array([offsets[k % 2], 0.0, 0.0])
    tp, bp = np.full(7, 1.0), np.full(6, 1.0)
    tp[2], tp[4], bp[1] = 30.0, 25.0, 30.0
    weight = rng.normal(size=6 * 7 * 8)
    got = api.ap_score_gradients(
        api.make_grid(res, lengths=lengths), api.Rational(api.POLYNOMIAL_4D(tr, tp, 1.1), api.POLYNOMIAL_4D(br, bp, 0.9)),
        api.make_params(1, 20.0, 0.8, 0.0, MAP_SKIP_ORIGIN | MAP_ADAPTIVE), api.make_grid((6, 7, 8), lengths=lengths),
        torch.from_numpy(weight).cuda(), 0.02, 0.1)
    ref = O.ap_score_gradients(
        og, O.poly(tr, tp, 1.1), O.poly(br, bp, 0.9),
        O.make_params(1, 20.0, 0.8, 0.0, O.SKIP_ORIGIN | O.AP_REPASS),
        O.make_grid((6, 7, 8), (0.0, 0.0, 0.0), lengths), weight, 0.02, 0.1)
    print(got["adaptive_cells"], ref["overflowed"], flush=True)
    assert got["adaptive_cells"] == ref["overflowed"]
    for k in ("score", "grad_exp", "grad_top", "grad_bottom", "grad_top_scalar", "grad_bottom_scalar"):
        a, b = np.atleast_1d(got[k]), np.atleast_1d(ref[k])
        assert np.max(np.abs(a - b)) <= 1e-9 * np.max(np.abs(b)), k
    assert np.allclose(got["field"].cpu().numpy(), ref["field"], rtol=1e-9, atol=1e-11)
