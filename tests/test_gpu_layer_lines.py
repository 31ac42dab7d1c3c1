"""The inverted distance's layer passes with the longest lines that a block holds
in LDS (512 cells, 16 lines along y and z: 64 KiB and the reduction's 8 KiB),
lines of some hundred cells and the first lengths beyond, along each axis. Layer
numbers and the plain inverted field bit for bit, the sum within n 2^-52
relative (double-double against the exact sum)."""
import math

import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [(3, 512, 2), (2, 3, 512), (19, 512, 3), (18, 3, 512), (5, 300, 400), (3, 513, 2),
                                 (2, 3, 513), (512, 5, 2)])
def test_long_lines(gpu, res):
    rng = np.random.default_rng(res[1])
    d = np.ones(res[0] * res[1] * res[2])
    d[rng.integers(0, d.size, 3)] = -2.0
    d[rng.integers(0, d.size, 5)] = 0.0
    lengths = tuple(0.1 * n for n in res)
    got, total = api.inverted_distance(torch.from_numpy(d).cuda(), api.make_grid(res, lengths=lengths))
    ref, _ = O.inverted_distance(O.make_grid(res, (0.0, 0.0, 0.0), lengths), d)
    assert np.array_equal(got.cpu().numpy(), ref)
    exact = math.fsum(np.abs(ref))
    assert abs(total - exact) <= d.size * 2.0 ** -52 * exact
