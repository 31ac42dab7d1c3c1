"""A workspace's first marching cubes call that fails for memory leaves nothing behind:
the next call, and torch's, are right."""
import numpy as np
import pytest
import torch

import oracle as O
from quijibo_amd import api
from quijibo_amd._lib import QJError

pytestmark = pytest.mark.gpu


def _too_many(n):
    """tiles whose vertices would take more than the card holds"""
    return int(2 * torch.cuda.get_device_properties(0).total_memory / (6 * n)) + 1


def test_call_after_a_failed_call(gpu):
    res = (64, 64, 96)
    n = res[0] * res[1] * res[2]
    f = np.random.default_rng(2).normal(size=n)
    d = torch.from_numpy(f).cuda()
    g = api.make_grid(res, lengths=(3.0, 3.0, 3.0))
    ws = api.Workspace()
    with pytest.raises(QJError):
        api.marching_cubes_tiles([d] * _too_many(n), [g] * _too_many(n), workspace=ws)
    assert float((d * 0.0).sum()) == 0.0
    with pytest.raises(QJError):
        api.marching_cubes_tiles([d] * _too_many(n), [g] * _too_many(n), workspace=ws)
    v, t = api.marching_cubes(d, g, workspace=ws)
    ov, ot = O.marching_cubes(O.make_grid(res, (0.0, 0.0, 0.0), (3.0, 3.0, 3.0)), f)
    assert np.array_equal(t, ot) and np.array_equal(v, ov)


def test_call_on_another_stream_after_a_failed_first_call(gpu):
    """The counters by which the kernels' last blocks are found are clear whatever
    the first call's stream still has to do."""
    res = (64, 64, 96)
    n = res[0] * res[1] * res[2]
    f = np.random.default_rng(3).normal(size=n)
    d = torch.from_numpy(f).cuda()
    g = api.make_grid(res, lengths=(3.0, 3.0, 3.0))
    ws = api.Workspace()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        x = torch.ones(1 << 26, device="cuda")
        for _ in range(200):
            x = x * 1.0001
    with pytest.raises(QJError):
        api.marching_cubes_tiles([d] * _too_many(n), [g] * _too_many(n), workspace=ws, stream=a)
    v, t = api.marching_cubes(d, g, workspace=ws, stream=b)
    ov, ot = O.marching_cubes(O.make_grid(res, (0.0, 0.0, 0.0), (3.0, 3.0, 3.0)), f)
    assert np.array_equal(t, ot) and np.array_equal(v, ov)
    torch.cuda.synchronize()
