"""qj_math64.h's functions on the device, through the calls that use them, over
their ranges: octants and quadrants with their edges, both ends, exponents whose
angle leaves the short reduction's range. References in 80-bit long double."""
import numpy as np
import pytest
import torch

import oracle as O
import test_gpu_adjoint_paths as adjoint
from quijibo_amd import api
from quijibo_amd._lib import FP64, FP64_EXACT, MAP_EXTENDED_RANGE

pytestmark = pytest.mark.gpu
LD = np.longdouble
NONE = np.zeros((0, 4))


def _poly(root, e):
    return api.Rational(api.POLYNOMIAL_4D([root], [e]), api.POLYNOMIAL_4D(NONE, []))


def _ulp(x):
    return np.spacing(np.abs(np.asarray(x, dtype=np.float64)))


def test_log(gpu):
    """F = log|q| of one exponent-1 root at the origin and one iteration: log64 of
    a square that is exact (points of 25 bits). At most 1 ulp."""
    rng = np.random.default_rng(0)
    m = np.concatenate([1 + np.arange(2049) / 2048, 1 + rng.integers(0, 1 << 24, 40000) / 2.0 ** 24,
                        1 + np.arange(1, 3000) / 2.0 ** 24, 2 - np.arange(1, 3000) / 2.0 ** 24,
                        np.sqrt(0.5) * 2 + np.arange(-200, 200) / 2.0 ** 22])
    m = np.round(m * 2.0 ** 24) / 2.0 ** 24
    x = np.concatenate([m * 2.0 ** k for k in (-1, 0, 39, -30, -300)])
    pts = np.stack([x, np.zeros_like(x), np.zeros_like(x)], axis=1)
    F = api.points_eval(torch.from_numpy(pts).cuda(), _poly([0, 0, 0, 0], 1.0), api.make_params(1, 2.0 ** 41, 1.0, 0.0, 0),
                        FP64).cpu().numpy()
    ref = np.log(x.astype(LD))
    assert F[x == 1.0].tolist() == [0.0] * int((x == 1.0).sum())
    err = np.abs(F - ref)[x != 1.0] / _ulp(ref)[x != 1.0]
    print("log: %.3f ulp" % err.max(), flush=True)
    assert err.max() <= 1.0


def test_tanh(gpu):
    """A weight score over one cell of weight 1 is -tanh(alpha (F - threshold)).
    At most 1 ulp, the bound of the library function it stands for."""
    rng = np.random.default_rng(1)
    x = np.concatenate([rng.uniform(-22, 22, 30000), rng.uniform(-1, 1, 30000), 2.0 ** rng.uniform(-60, 1, 20000),
                        np.arange(-40, 41) * 0.34657359027997264 / 2, [0.0, -0.0, 30.0, -700.0, 1e300, np.inf, -np.inf, 5e-324]])
    g = api.make_grid((1, 1, 1), lengths=(1.0, 1.0, 1.0))
    one, zero = torch.ones(1, dtype=torch.float64, device="cuda"), torch.zeros(1, dtype=torch.float64, device="cuda")
    parts = [api.weight_scores(zero, g, one, g, 1.0, p) for p in np.array_split(x, 2)]  # 1 (0 - x): -tanh(-x)
    sc = np.concatenate([p[0] for p in parts])
    assert all(p[1] == 1.0 for p in parts)
    ref = np.tanh(x.astype(LD))
    err = np.abs(sc - ref) / _ulp(ref)
    print("tanh: %.3f ulp" % err.max(), flush=True)
    assert err.max() <= 1.0


def _polar(b, e):
    """b^e of QUATERNION::pow in long double: unit part's and magnitude's product, and the angle"""
    b = b.astype(LD)
    v = np.sqrt(b[:, 1] ** 2 + b[:, 2] ** 2 + b[:, 3] ** 2)
    n = np.sqrt(v ** 2 + b[:, 0] ** 2)
    m = LD(e) * np.where(v > 0, np.arctan2(v, b[:, 0]), LD(0))
    f = np.where(v > 0, np.sin(m) / np.where(v > 0, v, LD(1)), LD(0))
    mag = np.exp(LD(e) * np.log(n))
    return np.concatenate([np.cos(m)[:, None], f[:, None] * b[:, 1:]], axis=1) * mag[:, None], m, n


def _directions(rng):
    """unit (w, |v|) pairs: random, the octants' edges (tan(pi/8), 1, the axes) and their neighbours"""
    a = [0.0, np.pi / 8, np.pi / 4, 3 * np.pi / 8, np.pi / 2, 5 * np.pi / 8, 3 * np.pi / 4, 7 * np.pi / 8, np.pi]
    ang = np.concatenate([rng.uniform(0, np.pi, 4000)] + [np.clip(c + s * 2.0 ** -np.arange(3.0, 60.0, 3.0), 0, np.pi)
                                                           for c in a for s in (-1, 1)])
    return np.cos(ang), np.sin(ang)


@pytest.mark.parametrize("e", [0.5, 0.7, 1.5, 3.0, 4.0, 7.3, 20.0])
@pytest.mark.parametrize("ext", [0, MAP_EXTENDED_RANGE])
def test_polar_power(gpu, e, ext):
    """Two iterations of one root: F = e log|b^e - r|, b = q - r. With u = 2^-53,
    b^e is off by at most |b^e| u (8 + 2 e + 3 |m| + 3 |e log|b||): |b|^2 off by 2 u,
    angle 2.5 ulp and log 0.9 ulp times e with the roundings of the products,
    exponential, sine and cosine within 1.3 ulp, |v| and 1 / |v| within 1.7; F then
    by e |b^e| / |b^e - r| of that and its own roundings."""
    rng = np.random.default_rng(2)
    c, s = _directions(rng)
    rad = np.exp(rng.uniform(-1.0, 1.0, len(c)))
    phi = rng.uniform(0, 2 * np.pi, len(c))
    root = np.array([0.25, -0.5, 0.125, 0.0])
    pts = root[:3] + np.stack([rad * c, rad * s * np.cos(phi), rad * s * np.sin(phi)], axis=1)
    b = np.concatenate([pts, np.zeros((len(pts), 1))], axis=1) - root  # rounded as the device rounds it
    q1, m, n = _polar(b, e)
    d = np.sqrt(((q1 - root) ** 2).sum(axis=1))
    ref = LD(e) * np.log(d)
    # within the escape radius; outside the extended range |b^e - r|^(2 e) in FP64's range
    use = np.asarray((np.sqrt((q1 ** 2).sum(axis=1)) < 1e11) & ((np.abs(ref) < 350) | (ext != 0)))
    F = api.points_eval(torch.from_numpy(pts).cuda(), _poly(root, e), api.make_params(2, 2.0 ** 40, 1.0, 0.0, ext),
                        FP64).cpu().numpy()
    u = 2.0 ** -53
    mag = np.sqrt((q1 ** 2).sum(axis=1))
    tol = e * mag / d * u * (8 + 2 * e + 3 * np.abs(m) + 3 * np.abs(e * np.log(n))) + 4 * u * (e + np.abs(ref))
    err = np.abs(F - ref) / tol
    print("e %g ext %d: %.3f of the bound" % (e, ext, err[use].max()), flush=True)
    assert use.sum() > 3000 and err[use].max() <= 1.0


@pytest.mark.parametrize("e", [3.0e8, 5.0e8, 1.3e9, 2.0e9, 3.1e9])
def test_polar_power_of_large_exponents(gpu, e):
    """The same with |b| next to 1 and an angle beyond 2^30, in the extended range
    (F = e log|b^e - r| is past FP64's range of the plain products)."""
    rng = np.random.default_rng(3)
    ang = rng.uniform(0.05, 3.0, 300)
    root = np.array([0.25, -0.5, 0.125, 0.0])
    pts = root[:3] + np.stack([np.cos(ang), np.sin(ang) * 0.6, np.sin(ang) * 0.8], axis=1)
    b = np.concatenate([pts, np.zeros((len(pts), 1))], axis=1) - root
    q1, m, n = _polar(b, e)
    d = np.sqrt(((q1 - root) ** 2).sum(axis=1))
    ref = LD(e) * np.log(d)
    F = api.points_eval(torch.from_numpy(pts).cuda(), _poly(root, e), api.make_params(2, 2000.0, 1.0, 0.0, MAP_EXTENDED_RANGE),
                        FP64).cpu().numpy()
    u = 2.0 ** -53
    mag = np.sqrt((q1 ** 2).sum(axis=1))
    # to second order: the shift of b^e stays a small part of its distance to the root
    shift = mag * u * (8 + 2 * e + 3 * np.abs(m) + 3 * np.abs(e * np.log(n)))
    use = np.asarray(shift < 0.01 * d)
    err = np.abs(F - ref) / (1.1 * e * shift / d + 4 * u * (e + np.abs(ref)))
    print("e %g: %d points, %.3f of the bound" % (e, use.sum(), err[use].max()), flush=True)
    assert use.sum() > 100 and err[use].max() <= 1.0


@pytest.mark.parametrize("e", [5.0e8, 1.3e9, 3.1e9])
def test_adjoint_of_large_exponents(gpu, e):
    """The same angles in the adjoint, against autograd: one term's gradient is off by
    its angle's error, 3 |m| 2^-53 < 3e-6, over the distance of b^e to the root."""
    rng = np.random.default_rng(5)
    ang = rng.uniform(0.3, 3.0, 64)
    root = np.array([[0.25, -0.5, 0.125, 0.0]])
    pts = root[0, :3] + np.stack([np.cos(ang), np.sin(ang) * 0.6, np.sin(ang) * 0.8], axis=1)
    g = rng.normal(size=len(pts))
    power = np.array([e])
    gr, gp = adjoint._reference(pts, root, power, NONE, np.zeros(0), g, 2, 1.0, 20.0)
    a, b = api.points_adjoint(torch.from_numpy(pts).cuda(), _poly(root[0], e), api.make_params(2, 20.0, 1.0, 0.0, 0),
                              torch.from_numpy(g).cuda(), FP64)
    ea = np.linalg.norm(a.cpu().numpy() - gr) / np.linalg.norm(gr)
    eb = np.linalg.norm(b.cpu().numpy() - gp) / np.linalg.norm(gp)
    print("e %g: %.2e %.2e" % (e, ea, eb), flush=True)
    assert ea <= 1e-3 and eb <= 1e-3


@pytest.mark.parametrize("iters", [1, 2])
@pytest.mark.parametrize("prec", [FP64, FP64_EXACT])
def test_bases_out_of_range(gpu, prec, iters):
    """Real powers of bases whose square is 0 or infinite in FP64 are not finite,
    as QUATERNION::pow's are (its |b| is 0 or infinite); the extended range takes
    them. Beside them bases whose squares are just inside."""
    s = np.array([1e-170, 3e-163, 1e-150, 1e-100, 1e-3, 0.5, 1e100, 1e150, 1e155, 1e200, 1e300])
    pts = np.concatenate([s[:, None] * d for d in np.array([[1.0, 0.5, -0.25], [0.0, 1.0, 0.0], [-1.0, 1e-3, 0.0],
                                                            [1.0, 1e-60, 0.0]])])
    for e in (0.003, 0.4, 1.5):
        gp = api.make_params(iters, np.inf, 1.0, 0.0, 0)
        F = api.points_eval(torch.from_numpy(pts).cuda(), _poly([0, 0, 0, 0], e), gp, prec).cpu().numpy()
        ref = O.points_eval(pts, O.poly([[0, 0, 0, 0]], [e]), O.poly(NONE, []), O.make_params(iters, np.inf, 1.0, 0.0, 0))
        assert np.array_equal(np.isfinite(F), np.isfinite(ref)), (e, pts[np.isfinite(F) != np.isfinite(ref)])
        fin = np.isfinite(ref)
        assert np.max(np.abs(F[fin] - ref[fin]) / np.maximum(1.0, np.abs(ref[fin]))) <= 1e-9
