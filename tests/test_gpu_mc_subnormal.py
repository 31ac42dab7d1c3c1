"""Marching cubes where the corner values are subnormal as floats: a vertex on a
grid point or next to it counts as near an end of its edge also where 1e-6 of
the values' difference is below the smallest float, so that the triangles that
shrink to a point are dropped as the oracle mesher drops them. Bit for bit."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values", [
    (0.0, 1e-42), (0.0, 1e-42, -1e-42), (0.0, 3e-45, -2e-44, 7e-40, -9e-41), (0.0, 1e-42, -3e-39, 1e-6, -1.0),
])
@pytest.mark.parametrize("lengths", [(1.0, 1.1, 0.9), (40.0, 30.0, 50.0), (3e-4, 3e-4, 4e-4)])
def test_subnormal_corners(gpu, lengths, values):
    res = (21, 18, 25)
    rng = np.random.default_rng(len(values))
    f = rng.choice(values, size=res[0] * res[1] * res[2])
    rotation = (0.8, 0.36, 0.48, 0.0)
    v, t = api.marching_cubes(torch.from_numpy(f).cuda(), api.make_grid(res, (0.1, 0.2, -0.1), lengths, rotation))
    ov, ot = O.marching_cubes(O.make_grid(res, (0.1, 0.2, -0.1), lengths, rotation), f)
    print(lengths, values, len(v), len(t), len(ot), flush=True)
    assert t.shape == ot.shape and np.array_equal(t, ot)
    assert v.shape == ov.shape and ((v == ov) | (np.isnan(v) & np.isnan(ov))).all()
