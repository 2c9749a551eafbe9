"""CPU check of the differentiated polynomials' coefficient map (mbx_amd/csrc/ad_slot.hpp), built for the
host: every slot is the exact combination of the fitted coefficients rounded once, and every second slot
what that rounding left."""
import os
import subprocess
import sys
from fractions import Fraction

import numpy as np
import pytest

from conftest import ROOT

sys.path.insert(0, ROOT + "/mbx_amd/gen")
import polygen  # noqa: E402


@pytest.mark.parametrize("coefficients", ["fitted", "random"])
@pytest.mark.parametrize("name", ["mbpol_2b", "mbpol_3b"])
def test_slots_are_rounded_once(name, coefficients, tmp_path):
    inc = os.path.join(ROOT, "mbx_amd", "csrc", "gen", "sym_%s.inc" % name)
    if not os.path.exists(inc):
        pytest.skip("the coefficient maps are generated by the build")
    _, fit, sym = polygen.adapted(name)
    a = np.array(fit)
    if coefficients == "random":
        rng = np.random.default_rng(4)
        a = rng.normal(size=len(a)) * 10.0 ** rng.uniform(-6, 6, len(a))
    a.tofile(tmp_path / "coef")
    program = str(tmp_path / "slots")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-I" + os.path.join(ROOT, "tests", "cpp", "host"),
                    "-DNAME=" + name, '-DSYM_INC="%s"' % inc, "-o", program,
                    os.path.join(ROOT, "tests", "cpp", "ad_slot_host.cpp")], check=True)
    out = subprocess.run([program, str(tmp_path / "coef")], check=True, capture_output=True, text=True).stdout
    slots = [float.fromhex(v) for v in out.split()]
    nrow = len(sym.rows)
    assert len(slots) == nrow + len(sym.low)
    exact = [sum(Fraction(float(a[k])) * Fraction(w) for k, w in r) for r in sym.rows]
    assert slots[:nrow] == [float(v) for v in exact]  # float() of a fraction rounds to nearest
    for j, q in enumerate(sym.low):
        size = sum(abs(Fraction(float(a[k])) * Fraction(w)) for k, w in sym.rows[q])
        # the rest is itself a sum of rounding errors, each below 2^-53 of a term and rounded at 2^-53 of that
        bound = size * len(sym.rows[q]) * Fraction(1, 2 ** 103)
        assert abs(Fraction(slots[nrow + j]) - (exact[q] - Fraction(slots[q]))) <= bound
