"""The polynomial of the complex-symmetric exponential (ctemsoft_amd/csrc/ctem_symcoef.h): its expansion from
the FP32 coefficients that the kernel takes."""
import math
import os
import subprocess

from numpy.polynomial import polynomial as P

from conftest import REPO


def _coefficients(tmp_path):
    exe = str(tmp_path / "symcoef_check")
    src = os.path.join(REPO, "tests", "native", "symcoef_check.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", src, "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()
    v = [float.fromhex(x) for x in out]
    return [complex(v[2 * i], v[2 * i + 1]) for i in range(6)]


def test_matches_exp_through_degree_seven(tmp_path):
    c, d1, d2, r, e1, g = _coefficients(tmp_path)
    b2 = [0, 0, 1]
    w = P.polyadd(P.polymul([0, c, 1], [0, c, 1]), P.polymul([d1], b2))
    x = P.polymul([r], P.polyadd(w, [0, d2]))
    p = P.polyadd(P.polyadd(P.polymul(x, x), P.polymul([e1], w)), P.polyadd(P.polymul([g], b2), [0, 1]))
    err = [p[k] * math.factorial(k) - 1 for k in range(9) if k]
    print(["%.1e" % abs(e) for e in err], "constant", p[0])
    # no constant, B exactly, B^2 to the rounding of g; the others carry a few FP32 roundings of the coefficients, whose
    # terms are up to four times their sum
    assert p[0] == 0 and err[0] == 0
    assert abs(err[1]) <= 2.0 ** -24
    assert max(abs(e) for e in err[2:7]) <= 16 * 2.0 ** -24
    assert abs(err[7]) < 0.75
    assert len(p) == 9

