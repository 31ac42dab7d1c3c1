"""Gradients of leaves on the host: each one owns its memory (exact comparisons)."""
import numpy as np
import pytest
import torch

from quijibo_amd import api, grad as G
from quijibo_amd._lib import MAP_BLACK_HOLE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("nt,nb", [(5, 3), (4, 0), (1, 1)])
def test_host_gradients_share_no_storage(gpu, nt, nb, dtype):
    rng = np.random.default_rng(nt)
    pts = torch.tensor(rng.uniform(-1.0, 1.0, (300, 3)), device="cuda")
    shapes = [(nt, 4), (nt,), (nb, 4), (nb,)]
    leaves = [torch.tensor(rng.uniform(0.5, 1.0, s), dtype=dtype, requires_grad=True) for s in shapes]
    F = G.julia_field(pts, *leaves, api.make_params(2, 2000.0, 1.0, 0.0, MAP_BLACK_HOLE))
    grads = torch.autograd.grad(F, leaves, torch.ones_like(F))
    for g, leaf in zip(grads, leaves):
        assert g.shape == leaf.shape and g.dtype == dtype and not g.is_cuda
        assert g.untyped_storage().nbytes() == g.numel() * g.element_size()
    used = [g.untyped_storage().data_ptr() for g in grads if g.numel()]
    assert len(set(used)) == len(used)
