"""Marching cubes where the degenerate filter measures vertices (spacings beyond the
prefilter's, coordinates beyond the estimates'): dense and sparse candidates, blocks
of 4 to 32 words with ragged ends, and fields beyond 512 groups, which measure in
the counting kernel. Bit for bit against the oracle mesher."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api

pytestmark = pytest.mark.gpu


def _field(kind, n, rng):
    if kind == "noise":
        return rng.normal(size=n)
    if kind == "binary":
        return (rng.random(n) < 0.5) * 1.0
    f = np.where(rng.random(n) < 0.002, 1.0, -1.0)  # isolated points, some next to grid points
    f[rng.integers(0, n, n // 500 + 1)] = 1e-9
    return f


@pytest.mark.parametrize("res, kind", [
    ((2, 2, 2), "binary"), ((5, 9, 3), "noise"), ((24, 23, 25), "binary"), ((65, 64, 63), "noise"),
    ((65, 64, 63), "sparse"), ((97, 101, 89), "binary"), ((129, 127, 130), "sparse"), ((163, 162, 161), "sparse"),
    ((163, 162, 161), "binary"), ((209, 203, 202), "sparse"),
])
def test_measured_cells(gpu, res, kind):
    n = res[0] * res[1] * res[2]
    f = _field(kind, n, np.random.default_rng(n))
    d = torch.from_numpy(f).cuda()
    for center, spacing in (((0.0, 0.0, 0.0), 4.0), ((3e4, 0.0, -1e4), 1.0), ((0.0, 0.0, 0.0), 3e-7)):
        lengths = tuple(spacing * r for r in res)
        v, t = api.marching_cubes(d, api.make_grid(res, center, lengths))
        ov, ot = O.marching_cubes(O.make_grid(res, center, lengths), f)
        print(res, kind, center, spacing, len(v), len(t), flush=True)
        assert t.shape == ot.shape and np.array_equal(t, ot)
        assert np.array_equal(v, ov)
