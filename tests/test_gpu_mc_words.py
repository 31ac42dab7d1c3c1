"""Marching cubes on bit words of 64 points: sizes around the word, the 256-cell
block and the 16384-point group, rows shorter and longer than a word, and
vertices at 1e-9 to 1e-4 spacings from grid points, where the degenerate filter
is decided by estimates, by measurement or not at all. Vertices, triangles and
their order must be those of the oracle mesher, bit for bit."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api

pytestmark = pytest.mark.gpu

RES = [(2, 2, 2), (2, 3, 70), (64, 2, 2), (65, 5, 3), (63, 64, 5), (128, 3, 4), (7, 9, 300), (1000, 3, 3),
       (64, 64, 9), (31, 33, 35)]


def field_of(kind, n, rng):
    sign = np.where(rng.random(n) < 0.5, -1.0, 1.0)
    if kind == "random":
        return sign * rng.random(n)
    if kind == "sparse":  # a few isolated points inside
        return np.where(rng.random(n) < 0.003, 1.0, -1.0)
    tiny = 10.0 ** rng.uniform(-9, -4, n)
    f = sign * np.where(rng.random(n) < 0.5, tiny, 1.0)
    f[rng.integers(0, n, n // 50 + 1)] = 0.0
    f[rng.integers(0, n, n // 90 + 1)] = np.inf
    f[rng.integers(0, n, n // 90 + 1)] = np.nan
    f[rng.integers(0, n, n // 90 + 1)] = 1e31
    f[rng.integers(0, n, n // 90 + 1)] = -1e-42
    return f


@pytest.mark.parametrize("kind", ["random", "sparse", "graded"])
@pytest.mark.parametrize("res", RES)
def test_words_match_the_oracle(gpu, res, kind):
    n = res[0] * res[1] * res[2]
    f = field_of(kind, n, np.random.default_rng(n + len(kind)))
    # spacings about 1; beyond the estimates' extent; below the prefilter's spacing
    for center, scale in (((0.1, -0.2, 0.3), 1.0), ((3e4, 0.0, -1e4), 1.0), ((0.0, 0.0, 0.0), 1e-7)):
        lengths = tuple(scale * r * (0.9 + 0.1 * i) for i, r in enumerate(res))
        rotation = (0.8, 0.36, 0.48, 0.0)
        v, t = api.marching_cubes(torch.from_numpy(f).cuda(), api.make_grid(res, center, lengths, rotation))
        ov, ot = O.marching_cubes(O.make_grid(res, center, lengths, rotation), f)
        print(res, kind, center, len(v), len(t), flush=True)
        assert v.shape == ov.shape and t.shape == ot.shape
        assert np.array_equal(t, ot)
        assert ((v == ov) | (np.isnan(v) & np.isnan(ov))).all()


@pytest.mark.parametrize("res", [(64, 64, 257), (128, 128, 1025)])
def test_group_scans(gpu, res):
    """65 groups (the tickets' second level) and 1025 (the scan of its own launch),
    twice in one workspace: the tickets are left as they were found."""
    n = res[0] * res[1] * res[2]
    f = field_of("sparse", n, np.random.default_rng(n))
    ov, ot = O.marching_cubes(O.make_grid(res, (0, 0, 0), (3, 3, 3), (1, 0, 0, 0)), f)
    ws, d = api.Workspace(), torch.from_numpy(f).cuda()
    for _ in range(2):
        v, t = api.marching_cubes(d, api.make_grid(res, (0, 0, 0), (3, 3, 3)), workspace=ws)
        assert np.array_equal(t, ot) and np.array_equal(v, ov)
