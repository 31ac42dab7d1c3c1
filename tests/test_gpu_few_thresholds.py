"""Weight scores of up to four thresholds (one pass) against the same thresholds
within a longer list (weights kept per cell) and the oracle: no threshold, one cell,
a block of 256 with a remainder, more cells than 1024 blocks take at once, fields
and weights that are not finite. The two routes' sums agree to the order of
double-double additions, 4 2^-53 of the absolute sum."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [(1, 1, 1), (257, 1, 1), (65, 64, 66), (31, 33, 35)])
@pytest.mark.parametrize("nthr", [0, 1, 2, 3, 4])
def test_few_thresholds(gpu, res, nthr):
    n = int(np.prod(res))
    rng = np.random.default_rng(n + nthr)
    f, w = rng.normal(size=n), rng.normal(size=6 * 5 * 4)
    g, og = api.make_grid(res, lengths=(2.0, 1.0, 1.5)), O.make_grid(res, (0.0, 0.0, 0.0), (2.0, 1.0, 1.5))
    wg, owg = api.make_grid((6, 5, 4), lengths=(1.8, 1.2, 1.5)), O.make_grid((6, 5, 4), (0.0, 0.0, 0.0), (1.8, 1.2, 1.5))
    thr = np.linspace(-1.0, 1.0, 6)
    F, Wt = torch.from_numpy(f).cuda(), torch.from_numpy(w).cuda()
    many, most = api.weight_scores(F, g, Wt, wg, 3.0, thr)
    few, mx = api.weight_scores(F, g, Wt, wg, 3.0, thr[:nthr])
    assert few.shape == (nthr,) and abs(mx - most) <= 4 * 2.0 ** -53 * most
    assert np.all(np.abs(few - many[:nthr]) <= 4 * 2.0 ** -53 * most)
    for k in range(nthr):
        rs, rm = O.weight_score(og, f, owg, w, 3.0, thr[k])
        assert abs(few[k] - rs) <= (n + 8) * 2.0 ** -52 * rm and abs(mx - rm) <= (n + 8) * 2.0 ** -52 * rm
    f[n // 2] = np.inf
    f[n // 3] = np.nan
    F = torch.from_numpy(f).cuda()
    many, _ = api.weight_scores(F, g, Wt, wg, 3.0, thr)
    few, _ = api.weight_scores(F, g, Wt, wg, 3.0, thr[:nthr])
    assert np.array_equal(np.isnan(few), np.isnan(many[:nthr]))
