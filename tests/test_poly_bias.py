"""CPU check that the generated polynomials have no error that adds up over n-mers.

The coefficients of the symmetry-adapted polynomials are rounded (mbx_amd/gen/symmetry.py), the same way in every n-mer; those
that matter carry a second coefficient with the rest.  The generated code, built for the host, is compared
with the exact coefficients in extended precision over liquid-like n-mers (the n-mers' own variables taken as exact): beside
what the coefficients without a second one leave, which is known, the mean error has to vanish within
five standard deviations of a mean.  And what they leave has to be the share that REST says."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT

sys.path.insert(0, ROOT + "/mbx_amd/gen")
import polygen  # noqa: E402
import symmetry  # noqa: E402

LD = np.longdouble
GEN = os.path.join(ROOT, "mbx_amd", "csrc", "gen")
N = 16384


@pytest.mark.parametrize("name, prefix", [("mbpol_2b", "poly_"), ("mbpol_3b", "poly_"), ("ch4h2o_2b", "poly_"),
                                          ("alkali_h2o2_3b", "xpoly_"), ("alkali_h2o_2b", "xpoly_"),
                                          ("co2co2_2b", "xpoly_")])
def test_no_error_that_adds_up(name, prefix, tmp_path):
    if not os.path.exists(os.path.join(GEN, "%s%s.inc" % (prefix, name))):
        pytest.skip("the untracked polynomials are generated by the build")
    nv, fit, sym = polygen.adapted(name)
    nrow = len(sym.rows)
    exact = [sum((LD(fit[k]) * LD(w) for k, w in r), LD(0)) for r in sym.rows]
    b = np.array([float(v) for v in exact])
    rest = np.array([float(v - LD(f)) for v, f in zip(exact, b)])
    x, _ = symmetry.sample_nmers(symmetry._HOLDERS.get(name, [name])[0], N)
    terms = [(q, m) for q, m in sym.terms if q < nrow]
    flat = np.zeros((len(terms), 10), np.int32)
    for row, (q, m) in zip(flat, terms):
        row[:2 + len(m)] = (q, len(m)) + tuple(m)
    path = tmp_path / "data"
    with open(path, "wb") as f:
        np.array([nv, N, nrow + len(sym.low), nrow, len(terms)], np.int32).tofile(f)
        for a in (x, b, rest[sym.low], rest, flat):
            np.ascontiguousarray(a).tofile(f)
    stub = tmp_path / "gen"
    stub.mkdir()
    fn = prefix + name
    text = open(os.path.join(GEN, fn + ".inc")).read().replace('#include "poly_support.hpp"', "")
    (stub / "poly.inc").write_text(text)
    program = str(tmp_path / "poly_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-march=native", "-ffp-contract=off", "-w", "-DPOLY=" + fn, "-DPARTS=1",
                    '-DPOLY_INC="%s"' % (stub / "poly.inc")] + (["-DENERGY_ONLY"] if "_e_parts" in text else [])
                   + ["-o", program, os.path.join(ROOT, "tests", "cpp", "poly_host.cpp")], check=True)
    out = subprocess.run([program, str(path)], check=True, capture_output=True, text=True).stdout
    # mean over the n-mers of every row's monomials and of their derivatives
    u = np.concatenate([sym.transform(x), np.ones((1, N))])
    mean = np.zeros((nrow, nv + 1))
    square = 0.0
    value = np.zeros((nrow, N))
    for q, m in terms:
        value[q] += np.prod(u[list(m)], axis=0)
        for i in range(len(m)):
            mean[q, m[i]] += np.prod(u[list(m[:i] + m[i + 1:])], axis=0).mean()
    mean[:, nv] = value.mean(axis=1)
    square = ((b[:, None] * value) ** 2).mean(axis=1).sum()
    left = rest.copy()
    left[sym.low] = 0.0
    kept = left @ mean
    assert abs(kept[nv]) <= 5 * symmetry.REST * 2.0 ** -53 * np.sqrt(square)
    for line in out.splitlines():
        parts, j, err, std = (float(v) for v in line.split())
        assert abs(err + kept[int(j)]) <= 5 * std / np.sqrt(N), (parts, j, err, kept[int(j)], std / np.sqrt(N))
