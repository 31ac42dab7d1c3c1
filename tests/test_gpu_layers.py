"""The inverted distance's layer passes at the sizes where they can go wrong: a
line of one cell, lines of 16, blocks of lines with a remainder, lines of
exactly the LDS limit (512) and beyond it, one sign change in a corner; and
weight scores with threshold counts around the kernel's four, saturated cells
and a weight grid of its own. Layer numbers and the plain inverted field bit for
bit, sums within n 2^-52 relative (double-double against the serial sums), the
scoring tests' own tolerances (tests/test_gpu_scoring.py)."""
import math

import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res, at", [
    ((2, 1, 1), (0, 0, 0)), ((16, 16, 16), (0, 0, 0)), ((17, 3, 5), (16, 2, 4)), ((5, 33, 18), (2, 16, 9)),
    ((512, 3, 2), (3, 1, 0)), ((513, 2, 3), (500, 0, 2)), ((2, 515, 3), (0, 7, 1)), ((3, 2, 600), (1, 1, 590)),
])
def test_layers_from_one_cell(gpu, res, at):
    d = np.ones(res[::-1])
    d[at[2], at[1], at[0]] = -2.0
    if d.size > 300:
        d[0, 0, res[0] // 2] = 0.0  # a zero has no shell of its own
    d = d.reshape(-1)
    lengths = tuple(0.1 * n for n in res)
    g, og = api.make_grid(res, lengths=lengths), O.make_grid(res, (0.0, 0.0, 0.0), lengths)
    got, total = api.inverted_distance(torch.from_numpy(d).cuda(), g)
    ref, _ = O.inverted_distance(og, d)
    rtotal = math.fsum(np.abs(ref))
    assert np.array_equal(got.cpu().numpy(), ref)
    tol = d.size * 2.0 ** -52
    assert abs(total - rtotal) <= tol * abs(rtotal)
    gn, a = api.inverted_distance(torch.from_numpy(d).cuda(), g, normalized=True)
    rn, ra = O.inverted_distance(og, d, normalized=True)
    assert np.max(np.abs(gn.cpu().numpy() - rn) / np.abs(rn)) <= tol and abs(a - ra) <= tol


@pytest.mark.parametrize("res, nthr", [((3, 2, 1), 1), ((7, 5, 9), 4), ((16, 16, 16), 5), ((40, 33, 50), 3)])
def test_weight_scores_threshold_counts(gpu, res, nthr):
    rng = np.random.default_rng(3 + nthr)
    n = int(np.prod(res))
    f = rng.normal(scale=3.0, size=n)  # alpha (F - t) saturates in most cells
    w = rng.normal(size=6 * 5 * 4)
    g, og = api.make_grid(res, lengths=(2.0, 1.0, 1.5)), O.make_grid(res, (0.0, 0.0, 0.0), (2.0, 1.0, 1.5))
    wg, owg = api.make_grid((6, 5, 4), lengths=(1.8, 1.2, 1.5)), O.make_grid((6, 5, 4), (0.0, 0.0, 0.0), (1.8, 1.2, 1.5))
    thr = np.linspace(-1.0, 1.0, nthr)
    sc, mx = api.weight_scores(torch.from_numpy(f).cuda(), g, torch.from_numpy(w).cuda(), wg, 10.0, thr)
    tol = n * 2.0 ** -52 + 4 * 2.0 ** -52  # the serial sum, and a few ulps of tanh per term
    for k, t in enumerate(thr):
        rs, rm = O.weight_score(og, f, owg, w, 10.0, t)
        assert abs(sc[k] - rs) <= tol * rm and abs(mx - rm) <= tol * rm
