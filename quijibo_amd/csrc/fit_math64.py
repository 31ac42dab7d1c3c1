"""Coefficients of the FP64 polynomials in qj_math64.h.

log     log(m) = 2 atanh(s) = 2 s + s z P(z), s = (m - 1) / (m + 1), z = s^2, m in [sqrt(1/2), sqrt(2)]
atan    atan(u) = u + u z P(z), z = u^2, |u| <= tan(pi / 8)
sin     sin(r) = r + r z P(z), z = r^2, |r| <= pi / 4
cos     cos(r) = 1 - z / 2 + z^2 P(z), the same range
exp     exp(r) = 1 + r + r^2 P(r), |r| <= ln 2 / 2 (z below is r itself)

Each P is the interpolant of its function at the Chebyshev nodes of its
interval in z, computed with 60 digits (mpmath) and rounded to FP64: within a
small factor of the minimax polynomial, which is far below an ulp here. Run as a
script to print the coefficients (lowest degree first).
"""


def _table():
    import mpmath as mp
    mp.mp.dps = 60

    def small(f, series):
        return lambda z: f(z) if z > mp.mpf(10) ** -12 else series(z)

    log = small(lambda z: (2 * mp.atanh(mp.sqrt(z)) / mp.sqrt(z) - 2) / z,
                lambda z: mp.mpf(2) / 3 + 2 * z / 5)
    atan = small(lambda z: (mp.atan(mp.sqrt(z)) / mp.sqrt(z) - 1) / z, lambda z: -mp.mpf(1) / 3 + z / 5)
    sin = small(lambda z: (mp.sin(mp.sqrt(z)) / mp.sqrt(z) - 1) / z, lambda z: -mp.mpf(1) / 6 + z / 120)
    cos = small(lambda z: (mp.cos(mp.sqrt(z)) - 1 + z / 2) / z ** 2, lambda z: mp.mpf(1) / 24 - z / 720)
    def exp(z):
        return (mp.exp(z) - 1 - z) / z ** 2 if abs(z) > mp.mpf(10) ** -12 else mp.mpf(1) / 2 + z / 6
    top = mp.sqrt(2)
    half = mp.log(2) / 2
    return {"log": (log, 0, ((top - 1) / (top + 1)) ** 2, 7), "atan": (atan, 0, mp.tan(mp.pi / 8) ** 2, 12),
            "sin": (sin, 0, (mp.pi / 4) ** 2, 6), "cos": (cos, 0, (mp.pi / 4) ** 2, 6),
            "exp": (exp, -half, half, 11)}


def coefficients(name):
    """The n coefficients of P, lowest degree first, as Python floats."""
    import mpmath as mp
    f, low, top, n = _table()[name]
    z = [low + (top - low) * (1 + mp.cos((2 * k + 1) * mp.pi / (2 * n))) / 2 for k in range(n)]
    a = mp.matrix(n, n)
    b = mp.matrix(n, 1)
    for i in range(n):
        b[i] = f(z[i])
        for j in range(n):
            a[i, j] = z[i] ** j
    c = mp.lu_solve(a, b)
    return [float(v) for v in c]


def max_error(name, points=400):
    """The largest |P - f| over the interval, relative to |f|, with exact evaluation of the rounded coefficients."""
    import mpmath as mp
    f, low, top, _ = _table()[name]
    c = [mp.mpf(v) for v in coefficients(name)]
    worst = mp.mpf(0)
    for k in range(1, points + 1):
        z = low + (top - low) * k / points
        p = mp.mpf(0)
        for v in reversed(c):
            p = p * z + v
        worst = max(worst, abs(p / f(z) - 1) * abs(z))
    return float(worst)


if __name__ == "__main__":
    for name in ("log", "atan", "sin", "cos", "exp"):
        print(name, [repr(v) for v in coefficients(name)], "rel err of the correction x z: %.2e" % max_error(name))
