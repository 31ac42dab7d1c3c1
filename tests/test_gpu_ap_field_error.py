"""The AP pass's field where top and bottom cancel: 8 + 8 roots at a distance of
e^5 with exponent 4, F = sum of terms of 20 and -20, near 0. The roots are taken in
turn from top and bottom, so that no running sum grows to 160 and back.

Root mean square bound, u = 2^-53 and a rounding of a value v off by 0.58 u 2^k
(2^k <= v): 16 logarithms of 0.3 ulp (8 u) of 5 times 4 each, 16 terms of 20 (16 u):
sqrt(16 (9.6^2 + 9.3^2)) u = 5.9e-15, and a third for what varies. Top roots first
and bottom roots last took 1.45e-14, the products of the formulas 4.2e-15."""
import numpy as np
import pytest
import torch

from quijibo_amd import api
from quijibo_amd._lib import MAP_ADAPTIVE, MAP_SKIP_ORIGIN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [(16, 15, 14), (33, 32, 34)])
def test_cancelling_sums(gpu, res):
    rng = np.random.default_rng(12)
    roots = rng.normal(size=(16, 4))
    roots *= np.exp(5.0) / np.linalg.norm(roots, axis=1, keepdims=True)
    lengths = (1.0, 1.25, 0.75)
    got = api.ap_score_gradients(
        api.make_grid(res, lengths=lengths),
        api.Rational(api.POLYNOMIAL_4D(roots[:8], np.full(8, 4.0)), api.POLYNOMIAL_4D(roots[8:], np.full(8, 4.0))),
        api.make_params(1, 20.0, 1.0, 0.0, MAP_SKIP_ORIGIN | MAP_ADAPTIVE), api.make_grid((4, 4, 4), lengths=lengths),
        torch.ones(64, dtype=torch.float64, device="cuda"), 2.0, 0.1)
    ax = [-0.5 * l + (np.arange(n) + 0.5) * (l / n) for n, l in zip(res, lengths)]
    Z, Y, X = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    q = np.stack([X.reshape(-1), Y.reshape(-1), Z.reshape(-1), 0 * X.reshape(-1)], axis=1).astype(np.longdouble)
    F = sum((1 if i < 8 else -1) * 2 * np.log(((q - r) ** 2).sum(axis=1)) for i, r in enumerate(roots))
    err = got["field"].cpu().numpy() - F
    near = np.sqrt((q ** 2).sum(axis=1)) > 1e-8
    rms = float(np.sqrt((err[near] ** 2).mean()))
    print("rms %.2e, F up to %.2f" % (rms, np.abs(F).max()), flush=True)
    assert rms <= 7.9e-15
