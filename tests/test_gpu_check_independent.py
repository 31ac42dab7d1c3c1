"""The sampled FP64 cross-check evaluates the map in polar form with the device
library's functions, in the reference's order: never by the code that wrote the
field. So on a field of QJ_FP64 or QJ_FP64_EXACT (exponents 1 and 2 as products,
the other powers from short functions, the last iteration from norms) it finds
rounding differences, which a check against itself would not.

Bounds: larger than 0, below 1e-9 max(1, |F|), the field tests' own
(tests/test_gpu_field.py), no sign flips and no class mismatch."""
import numpy as np
import pytest
import torch

from quijibo_amd import api, workloads as W
from quijibo_amd._lib import FP64, FP64_EXACT, MAP_BLACK_HOLE, MAP_EXTENDED_RANGE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("powers", ["int", "real"])
@pytest.mark.parametrize("flags", [MAP_BLACK_HOLE, MAP_BLACK_HOLE | MAP_EXTENDED_RANGE])
@pytest.mark.parametrize("prec", [FP64, FP64_EXACT])
def test_check_is_not_the_fields_own_evaluator(gpu, prec, flags, powers):
    w = W.config2(24)
    tp, bp = w.top.powers, w.bottom.powers
    if powers == "real":
        rng = np.random.default_rng(4)
        tp, bp = rng.uniform(0.4, 1.6, len(tp)), rng.uniform(0.4, 1.6, len(bp))
    g = api.make_grid(w.res, w.center, w.lengths)
    r = api.Rational(api.POLYNOMIAL_4D(w.top.roots, tp), api.POLYNOMIAL_4D(w.bottom.roots, bp))
    p = api.make_params(2, w.escape, w.exp_scaling, w.slice, flags)
    ws = api.Workspace()
    ws.check(w.voxels)
    ws.reset_stats()
    api.field_eval(g, r, p, prec, workspace=ws)
    st = ws.stats()
    print({k: st[k] for k in st if k.startswith("check")}, flush=True)
    assert st["checked"] == w.voxels
    assert st["check_sign_flips"] == 0 and st["check_class_mismatch"] == 0
    assert 0 < st["check_max_rel_dF"] < 1e-9
