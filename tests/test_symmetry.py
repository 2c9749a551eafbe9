"""CPU checks of the symmetry-adapted polynomials (mbx_amd/gen/symmetry.py).

With u the Walsh-Hadamard transform of x and b = T a (plus the second coefficients), the adapted
polynomial must have the table's value, and its gradient in u, transformed back, the table's gradient,
for any coefficients.  Both are summed in extended precision, so what is left is the rounding of u and b:
each term's few factors and the coefficient round by 2^-53, 16 x 2^-53 of the terms' magnitudes at most.
"""
import sys

import numpy as np
import pytest

from conftest import ROOT

sys.path.insert(0, ROOT + "/mbx_amd/gen")
import polygen  # noqa: E402
import symmetry  # noqa: E402

LD = np.longdouble


def value_and_gradient(terms, c, x):
    """(P, dP/dx, sum of the terms' magnitudes) of sum c[q] prod x[m], in extended precision."""
    p, g, scale = LD(0), np.zeros(len(x), LD), LD(0)
    x = np.asarray(x, LD)
    for q, m in terms:
        v = x[list(m)]
        t = LD(c[q]) * np.prod(v)
        p, scale = p + t, scale + abs(t)
        for i in m:
            g[i] += t / x[i]
    return p, g, scale


@pytest.mark.parametrize("name", sorted(symmetry.EXCHANGES))
def test_adapted_polynomial(name):
    nv, fit, sym = polygen.adapted(name)
    _, _, monos = polygen.load_table(name)
    if name == "ch4ch4_2b":  # a tenth of its 201,250 monomials' orbits, to keep the sum short
        keep = set(range(0, len(fit), 10))
        monos = [t for t in monos if t[0] in keep]
    rng = np.random.default_rng(8)
    x = rng.uniform(0.2, 1.4, nv)
    a = np.zeros(len(fit))
    used = sorted(set(k for k, _ in monos))
    a[used] = rng.normal(size=len(used)) * 10.0 ** rng.uniform(-3, 3, len(used))
    exact = [sum((LD(a[k]) * LD(w) for k, w in r), LD(0)) for r in sym.rows]
    b = [float(v) for v in exact]
    b += [float(exact[q] - LD(b[q])) for q in sym.low]
    p0, g0, scale = value_and_gradient(monos, a, x)
    p1, gu, _ = value_and_gradient([t for t in sym.terms if b[t[0]] != 0.0], b, sym.transform(x))
    g1 = sym.transform(gu)  # the transform is its own transpose
    tol = 16 * 2.0 ** -53 * float(scale)
    assert abs(float(p1 - p0)) <= tol
    np.testing.assert_allclose(np.asarray(g1 - g0, float), 0.0, atol=tol / x.min())
    # every monomial of the adapted polynomial once, and again for each second coefficient
    first = [m for q, m in sym.terms if q < len(sym.rows)]
    assert len(first) == len(set(first)) and len(first) < len(monos) or name == "ch4ch4_2b"


def test_exchange_that_is_no_symmetry_is_refused():
    nv, _, monos = polygen.load_table("mbpol_2b")
    with pytest.raises(ValueError):
        symmetry._check_invariant("mbpol_2b", nv, monos, [[1, 0] + list(range(2, nv))])
