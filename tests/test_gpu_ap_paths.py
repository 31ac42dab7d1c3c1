"""The AP pass's two routes at the sizes where they meet: blocks of 64 and of
256 cells with ragged ends, cells beyond the logarithms' range beside cells
within it, exponents of zero, and negative exponents (which take the general
route for every cell), against the oracle. Tolerance 1e-9 relative, the AP
pass's own (tests/test_gpu_grad.py)."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api
from quijibo_amd._lib import MAP_ADAPTIVE, MAP_SKIP_ORIGIN

pytestmark = pytest.mark.gpu


def _roots(rng, n):
    return np.concatenate([rng.normal(scale=0.6, size=(n, 3)), rng.uniform(-0.1, 0.1, size=(n, 1))], axis=1)


@pytest.mark.parametrize("res, nt, nb, powers", [
    ((3, 2, 2), 1, 0, "real"),         # one block, fewer roots than waves
    ((8, 4, 2), 5, 3, "real"),         # exactly one block of 64 cells
    ((13, 5, 1), 4, 9, "zero"),        # one cell into the second block; exponents of 0
    ((32, 32, 32), 3, 2, "real"),      # the first grid of 256-cell blocks
    ((33, 31, 35), 2, 3, "range"),     # ragged 256-cell blocks, some cells beyond the range
    ((9, 8, 7), 40, 26, "real"),       # more than 64 roots, both block sizes
    ((33, 32, 32), 40, 26, "real"),
    ((7, 5, 9), 140, 121, "small"),    # more than 256 roots
    ((9, 9, 9), 3, 3, "range"),        # 64-cell blocks, the origin cell, some cells beyond the range
    ((11, 7, 5), 4, 4, "negative"),    # the general route throughout
])
def test_ap_pass_routes(gpu, res, nt, nb, powers):
    rng = np.random.default_rng(71)
    tr, br = _roots(rng, nt), _roots(rng, nb)
    tp, bp = rng.uniform(0.4, 2.0, size=nt), rng.uniform(0.4, 2.0, size=nb)
    if powers == "small":
        tp, bp = 0.2 * tp, 0.2 * bp
    if powers == "zero":
        tp[1] = bp[2] = bp[5] = 0.0
    if powers == "range":  # 400 log|b| passes 340 in the box's corners only
        tp[0] = bp[0] = 400.0
    if powers == "negative":
        tp[1] = -0.7
    weight = rng.normal(size=6 * 7 * 8)
    lengths = (3.0, 2.5, 2.75)
    gpu_r = api.ap_score_gradients(
        api.make_grid(res, lengths=lengths),
        api.Rational(api.POLYNOMIAL_4D(tr, tp, 1.1), api.POLYNOMIAL_4D(br, bp, 0.9)),
        api.make_params(1, 20.0, 0.8, 0.0, MAP_SKIP_ORIGIN | MAP_ADAPTIVE), api.make_grid((6, 7, 8), lengths=lengths),
        torch.from_numpy(weight).cuda(), 2.0, 0.1)
    cpu = O.ap_score_gradients(
        O.make_grid(res, (0.0, 0.0, 0.0), lengths), O.poly(tr, tp, 1.1), O.poly(br, bp, 0.9),
        O.make_params(1, 20.0, 0.8, 0.0, O.SKIP_ORIGIN | O.AP_REPASS),
        O.make_grid((6, 7, 8), (0.0, 0.0, 0.0), lengths), weight, 2.0, 0.1)
    assert gpu_r["adaptive_cells"] == cpu["overflowed"]
    for k in ("score", "grad_exp", "grad_top", "grad_bottom", "grad_top_scalar", "grad_bottom_scalar"):
        a, b = np.atleast_1d(gpu_r[k]), np.atleast_1d(cpu[k])
        assert a.shape == b.shape
        if a.size:
            assert np.max(np.abs(a - b)) <= 1e-9 * max(1e-300, np.max(np.abs(b))), k
    assert np.allclose(gpu_r["field"].cpu().numpy(), cpu["field"], rtol=1e-9, atol=1e-12)
