"""The polynomials of qj_math64.h: their coefficients are the ones
quijibo_amd/csrc/fit_math64.py fits, and each is within 2^-53 of its function
as a correction to the leading term."""
import os
import re
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "quijibo_amd", "csrc")
sys.path.insert(0, CSRC)
pytest.importorskip("mpmath")
import fit_math64  # noqa: E402


@pytest.mark.parametrize("name, begins, ends", [
    ("log", "const double z = s * s;", "// f - R"),
    ("atan", "const double z = u * u;", "// +-(u + u z P)"),
    ("sin", "double p = k64<kInLoop>(1.59", "const double s = "),
    ("cos", "double c = k64<kInLoop>(", "c = __builtin_fma(z, "),
    ("exp", "double p = k64<kInLoop>(2.09", "return p;"),
])
def test_constants_are_the_fit(name, begins, ends):
    src = open(os.path.join(CSRC, "qj_math64.h")).read()
    body = src[src.index(begins):]
    body = body[:body.index(ends)]
    first = re.search(r"double [pc] = k64<kInLoop>\(([-0-9.e]+)\);", body).group(1)
    rest = re.findall(r"__builtin_fma\([pc], [zr], k64<kInLoop>\(([-0-9.e]+)\)\)", body)
    got = [float(v) for v in [first] + rest][::-1]
    assert got == fit_math64.coefficients(name)
    assert fit_math64.max_error(name, 100) < 2.0 ** -53 * 1.1
