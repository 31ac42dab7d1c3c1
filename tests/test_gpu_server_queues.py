"""The request loop's work queues and band lists: chunks smaller than, equal to
and no multiple of a 256-voxel tile, fewer tiles than queues, requests of all
four FP32 variants in one launch, and a band that sends every voxel to the FP64
pass (each queue's part of the list filled to its end). Results must be those of
the direct evaluation bit for bit: batching changes no arithmetic."""
import numpy as np
import pytest

from quijibo_amd import api, server as S, workloads as W
from quijibo_amd._lib import FP32_BAND, FP64, MAP_BLACK_HOLE

pytestmark = pytest.mark.gpu


def requests(rng):
    out = []
    for i, res in enumerate([(3, 2, 2), (17, 9, 5), (40, 33, 21), (16, 16, 16), (31, 8, 9), (64, 5, 3)]):
        nt, nb = int(rng.integers(2, 9)), int(rng.integers(2, 9))
        kind = i % 4
        tp = rng.choice([1.0, 1.5, 2.0], size=nt) if kind == 2 else rng.integers(1, 3, size=nt).astype(float)
        if kind == 3:
            tp = np.ones(nt)
        out.append(W.Workload("q%d" % i, res, W.RootSet(rng.normal(scale=0.7, size=(nt, 4)), tp),
                              W.RootSet(rng.normal(scale=0.7, size=(nb, 4)), np.ones(nb)), max_iter=3,
                              escape=1e6 if kind == 1 else 2000.0))
    return out


@pytest.mark.parametrize("band", [0.05, 1e30])
@pytest.mark.parametrize("chunk,per_launch", [(37, 512), (255, 8), (256, 1), (257, 3), (1000, 64), (65536, 512)])
def test_queues_change_no_result(gpu, chunk, per_launch, band):
    reqs = requests(np.random.default_rng(chunk))
    for precision in (FP32_BAND, FP64):
        srv = S.Server(hbm_budget_bytes=256 << 20, chunk_voxels=chunk, chunks_per_launch=per_launch,
                       precision=precision, band=band)
        ids = [srv.submit(w, keep_field=True) for w in reqs]
        done = {c.id: c for c in srv.wait_all(len(reqs), timeout=60)}
        assert len(done) == len(reqs) and all(c.status == 0 for c in done.values())
        got = [srv.fetch(done[i], device=False) for i in ids]
        srv.close()
        for w, f in zip(reqs, got):
            r = api.Rational(api.POLYNOMIAL_4D(w.top.roots, w.top.powers),
                             api.POLYNOMIAL_4D(w.bottom.roots, w.bottom.powers))
            ref = api.field_eval(api.make_grid(w.res, w.center, w.lengths), r,
                                 api.make_params(w.max_iter, w.escape, w.exp_scaling, w.slice, MAP_BLACK_HOLE),
                                 precision, band).cpu().numpy()
            assert np.array_equal(ref.reshape(-1), np.asarray(f).reshape(-1), equal_nan=True), (w.name, precision)
