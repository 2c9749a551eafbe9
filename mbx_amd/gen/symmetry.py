"""Symmetry-adapted coordinates of the permutationally-invariant polynomials.

A polynomial of mbx_amd/tables is unchanged when like sites of one molecule are exchanged: the two
hydrogens of a water, its two lone-pair sites, the oxygens of a CO2, the hydrogens of a CH4 by
double transpositions.  Those exchanges commute and square to the identity, so they form a group G
of 2^m elements that permutes the variables, and every variable orbit (1 to 16 variables) has a
basis of sums and differences

    u_c = sum_e (-1)^(c . e) x_e            (a Walsh-Hadamard transform of the orbit)

each of which is multiplied by +1 or -1 under every element of G: its character.  A monomial in the
u is multiplied by the product of its factors' characters, so in these coordinates the invariant
polynomial holds only the monomials whose characters multiply to +1, about one in |G| of them:
the 33,525 monomials of the MB-pol 3B polynomial become 6,773, the 201,250 of CH4-CH4 15,235.  It
is the same polynomial with the same value; its gradient follows by the (symmetric) transform,
dE/dx = H dE/du.

The new coefficients are fixed linear combinations b = T a of the fitted ones, with dyadic weights.  Most
tables have as many distinct combinations as coefficients.  A combination rounds once, the same way in
every n-mer, so over many n-mers that error adds up where the others average out: 256 waters lose 2.5e-9
(2B) and 3.3e-9 (3B) kcal/mol to it, where the original coordinates are off by 4e-10 and 1e-10 either way.  It
comes from few combinations: those that matter most, for the monomials they cost, carry a second coefficient
with the rounded-off rest on the same monomials.  With REST of the error left 256 waters are off by some 2e-11
of that kind in each order, less than the random error of the largest boxes in use.
"""
import collections
import itertools
import json
import math
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
TABLES = os.path.join(os.path.dirname(HERE), "tables")

# Exchanges of like sites, as site swaps; the sites are those of the holder's variables (MB-pol: below).
_WATERS = {n: [[(3 * i + 1, 3 * i + 2)] for i in range(n)] for n in (2, 3, 4)}


def _methane(c):
    return [[(c + 1, c + 2), (c + 3, c + 4)], [(c + 1, c + 3), (c + 2, c + 4)]]


EXCHANGES = {
    "mbpol_2b": [[(1, 2)], [(4, 5)], [(6, 7)], [(8, 9)]],
    "mbpol_3b": _WATERS[3],
    "ch4h2o_2b": [[(1, 2)], [(8, 9)]] + _methane(3),
    "ch4ch4_2b": _methane(0) + _methane(5),
    "ch4h2o2_3b": _methane(0) + [[(6, 7)], [(9, 10)]],
    "halide_h2o_2b": [[(2, 3)], [(4, 5)]],
    "alkali_h2o_2b": [[(1, 2)], [(4, 5)]],
    "co2co2_2b": _WATERS[2],
    "halide_h2o2_3b": [[(2, 3)], [(5, 6)], [(7, 8)], [(9, 10)]],
    "alkali_h2o2_3b": _WATERS[2],
    "co2x3_3b": _WATERS[3],
    "h2ox4_4b": _WATERS[4],
}
# the holders of the structures that serve several
_HOLDERS = {s + t: [i + t for i in ions] for s, ions in (("halide", ("cl", "f", "br", "i")),
                                                         ("alkali", ("na", "li", "k", "rb", "cs")))
            for t in ("_h2o_2b", "_h2o2_3b")}

# MB-pol: (rate, offset, Coulomb-like) of each variable class (2B x2b-v9x.cpp:1330-1345, 3B x3b-v2x.cpp:1256-1271)
_MBPOL_CLASS = {
    "mbpol_2b": [(-0.648, 1.0, False), (1.675, 1.0, False), (1.148, 4.0, True), (1.206, 4.0, True), (1.395, 4.0, True),
                 (0.735, 4.0, False), (0.800, 4.0, False), (0.796, 4.0, False)],
    "mbpol_3b": [(-2.254, 1.691, False), (-0.256, -3.0, False), (0.425, 3.499, False), (0.813, 4.854, False),
                 (0.0375, 0.0, False)],
}

# MB-pol: (class, site, site) per variable; sites O H H per water, then (2B) each water's lone pairs
_MBPOL = {
    "mbpol_2b": [(0, 1, 2), (0, 4, 5), (1, 0, 1), (1, 0, 2), (1, 3, 4), (1, 3, 5), (2, 1, 4), (2, 1, 5), (2, 2, 4),
                 (2, 2, 5), (3, 0, 4), (3, 0, 5), (3, 3, 1), (3, 3, 2), (4, 0, 3), (5, 6, 4), (5, 6, 5), (5, 7, 4),
                 (5, 7, 5), (5, 8, 1), (5, 8, 2), (5, 9, 1), (5, 9, 2), (6, 0, 8), (6, 0, 9), (6, 3, 6), (6, 3, 7),
                 (7, 6, 8), (7, 6, 9), (7, 7, 8), (7, 7, 9)],
    "mbpol_3b": [(0, 1, 2), (0, 4, 5), (0, 7, 8), (1, 0, 1), (1, 0, 2), (1, 3, 4), (1, 3, 5), (1, 6, 7), (1, 6, 8),
                 (2, 1, 4), (2, 1, 5), (2, 1, 7), (2, 1, 8), (2, 2, 4), (2, 2, 5), (2, 2, 7), (2, 2, 8), (2, 4, 7),
                 (2, 4, 8), (2, 5, 7), (2, 5, 8), (3, 0, 4), (3, 0, 5), (3, 0, 7), (3, 0, 8), (3, 3, 1), (3, 3, 2),
                 (3, 3, 7), (3, 3, 8), (3, 6, 1), (3, 6, 2), (3, 6, 4), (3, 6, 5), (4, 0, 3), (4, 0, 6), (4, 3, 6)],
}


def _holder(name):
    with open(os.path.join(TABLES, _HOLDERS.get(name, [name])[0] + ".holder.json")) as f:
        return json.load(f)


# Sites of a molecule (Angstrom) and its centre's distance to a neighbour's, at least
_SHAPE = {
    "h2o": [(0.0, 0.0, 0.0), (0.757, 0.587, 0.0), (-0.757, 0.587, 0.0)],
    "ch4": [(0.0, 0.0, 0.0), (0.629, 0.629, 0.629), (0.629, -0.629, -0.629), (-0.629, 0.629, -0.629),
            (-0.629, -0.629, 0.629)],
    "co2": [(0.0, 0.0, 0.0), (1.16, 0.0, 0.0), (-1.16, 0.0, 0.0)],
}
_CONTACT = {"h2o": 2.5, "ch4": 3.4, "co2": 3.4}
_LONE_PAIR = (-0.0972, 0.0986)  # in the plane, out of it (x2b-v9x.cpp:1346-1347)


def sample_nmers(name, n):
    """(variables (nvars, n), switch (n)) of n-mers as a liquid has them: the molecules' centres anywhere
    around the first one that the switch and the neighbours leave, random orientations, vibrating bonds."""
    rng = np.random.default_rng(1)
    if name in _MBPOL:
        order = 3 if name == "mbpol_3b" else 2
        mols = ["h2o"] * order
        vs = [(k, d, f, a, b) for c, a, b in _MBPOL[name] for k, d, f in [_MBPOL_CLASS[name][c]]]
        inner, outer = (4.5, 6.5) if order == 2 else (0.0, 4.5)
        lone = [0, 3] if order == 2 else []
    else:
        h = _holder(name)
        mols = h["monomers"]
        vs = [(k, d if f in ("exp0", "coul0") else 0.0, f in ("coul0", "coul"), a, b) for f, k, d, a, b in h["vars"]]
        inner, outer = h["switch"]["inner"], h["switch"]["outer"]
        lone = [v["oxygen_site"] for v in (h["vsites"] if "vsites" in h else [h["vsite"]] if h.get("vsite") else [])]
    centres, count = [], 0
    while count < n:
        c = rng.uniform(-outer, outer, (8 * n, len(mols), 3))
        c[:, 0] = 0.0
        ok = np.ones(len(c), bool)
        far = np.zeros(len(c), int)
        for i in range(len(mols)):
            for j in range(i):
                r = np.linalg.norm(c[:, i] - c[:, j], axis=1)
                ok &= r > (_CONTACT.get(mols[i], 2.5) + _CONTACT.get(mols[j], 2.5)) / 2
                far += r > outer
        centres.append(c[ok & (far <= (len(mols) == 3))])  # three-body switches: sums over two of the pairs
        count += len(centres[-1])
    c = np.concatenate(centres)[:n]
    pairs = [(i, j) for i in range(len(mols)) for j in range(i)]
    sw = []
    for i, j in pairs:
        t = np.clip((np.linalg.norm(c[:, i] - c[:, j], axis=1) - inner) / (outer - inner), 0.0, 1.0)
        sw.append(0.5 * (1.0 + np.cos(np.pi * t)))
    weight = sw[0] * sw[1] + sw[0] * sw[2] + sw[1] * sw[2] if len(mols) == 3 else np.prod(sw, axis=0)
    sites = []
    for m, kind in enumerate(mols):
        body = np.array(_SHAPE.get(kind, [(0.0, 0.0, 0.0)]))
        q = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0]
        at = (body + rng.normal(0.0, 0.03, (n,) + body.shape) * (np.abs(body).sum(1) > 0)[:, None]) @ q
        sites += [c[:, m] + at[:, k] for k in range(len(body))]
    for o in lone:
        p, q = sites[o + 1] - sites[o], sites[o + 2] - sites[o]
        mid, out = sites[o] + 0.5 * _LONE_PAIR[0] * (p + q), _LONE_PAIR[1] * np.cross(p, q)
        sites += [mid + out, mid - out]
    x = []
    for k, d, coulomb, a, b in vs:
        r = np.linalg.norm(sites[a] - sites[b], axis=1)
        v = np.exp(k * (d - r))
        x.append(v / r if coulomb else v)
    return np.array(x), weight


def variable_permutations(name):
    """Each exchange as a permutation of the variables."""
    if name in _MBPOL:
        vs = [(c, frozenset((a, b))) for c, a, b in _MBPOL[name]]
    else:
        vs = [(tuple(v[:3]), frozenset(v[3:5])) for v in _holder(name)["vars"]]
    index = {v: i for i, v in enumerate(vs)}
    out = []
    for swaps in EXCHANGES[name]:
        to = {}
        for a, b in swaps:
            to[a], to[b] = b, a
        out.append([index[(c, frozenset(to.get(s, s) for s in p))] for c, p in vs])
    return out


def _key(rows, base):
    """Each row of small integers as one integer."""
    key = np.zeros(len(rows), np.int64)
    for d in range(rows.shape[1]):
        key = key * base + rows[:, d]
    return key


def _parity(v):
    return bin(v).count("1") & 1


# Share of the combinations' rounding error that may stay without a second coefficient.
REST = 1.0 / 60.0


class Adapted:
    """blocks: the variable orbits of 2 or more, in transform order; terms: [(slot, monomial in u)];
    rows[slot]: [(fitted coefficient index, weight)]; low: the slots whose rounded-off rest is slot
    len(rows) + position."""

    def __init__(self, name, nvars, monos, coef):
        perms = variable_permutations(name)
        _check_invariant(name, nvars, monos, perms)
        ng = len(perms)
        elements = []
        for mask in range(1 << ng):
            p = list(range(nvars))
            for b in range(ng):
                if mask >> b & 1:
                    p = [perms[b][i] for i in p]
            elements.append(p)
        self.nvars, self.blocks = nvars, []
        char = np.zeros(nvars, np.int64)              # character of u_i as a bit mask over the exchanges
        inv = [[(i, 1.0)] for i in range(nvars)]      # x_i as [(u, weight)]
        done = set()
        for i in range(nvars):
            if i in done:
                continue
            stab = [m for m in range(1 << ng) if elements[m][i] == i]
            reps = []                                 # exchanges that generate the orbit
            orbit = [i]
            for m in range(1 << ng):
                if elements[m][i] not in orbit:
                    orbit += [elements[m][v] for v in orbit]
                    reps.append(m)
            done.update(orbit)
            if len(orbit) == 1:
                continue
            self.blocks.append(orbit)
            for c, u in enumerate(orbit):
                # the character that is trivial on the stabiliser and (-1)^(bit j of c) on reps[j]
                char[u] = next(x for x in range(1 << ng) if not any(_parity(x & s) for s in stab)
                               and all(_parity(x & r) == (c >> j & 1) for j, r in enumerate(reps)))
            for e, v in enumerate(orbit):
                inv[v] = [(u, (-1.0 if _parity(c & e) else 1.0) / len(orbit)) for c, u in enumerate(orbit)]
        self._expand(monos, elements, char, inv)
        self._second_coefficients(name, coef)

    def transform(self, x):
        """u of the variables x (nvars, n)."""
        u = np.array(x)
        for orbit in self.blocks:
            step = 1
            while step < len(orbit):
                for i in range(len(orbit)):
                    if not i & step:
                        p, q = orbit[i], orbit[i + step]
                        u[p], u[q] = u[p] + u[q], u[p] - u[q]
                step *= 2
        return u

    def _second_coefficients(self, name, coef):
        """Terms for the rests of the combinations that carry all but REST of the rounding error, judged
        on sampled n-mers (of every holder that the structure serves)."""
        nrow = len(self.rows)
        count = np.bincount([q for q, _ in self.terms], minlength=nrow)
        rounded = np.array([len(r) > 1 or math.frexp(r[0][1])[0] not in (0.5, -0.5) for r in self.rows])
        share = np.zeros(nrow)
        for holder in _HOLDERS.get(name, [name]):
            a = _holder(holder)["coef"] if name in _HOLDERS else coef
            x, switch = sample_nmers(holder, 512)
            u = self.transform(x)
            size = np.zeros((nrow, u.shape[1]))
            for q, m in self.terms:
                size[q] += np.prod(u[list(m)], axis=0) if m else 1.0
            b = np.array([sum(a[k] * w for k, w in r) for r in self.rows])
            err = b ** 2 * ((size * switch) ** 2).mean(axis=1) * rounded  # a rounded b's, in units of 2^-53 / sqrt(3)
            share = np.maximum(share, err / err.sum())
        order = np.argsort(-share / count, kind="stable")
        left = np.cumsum(share[order][::-1])[::-1]  # what stays if order[i:] have none
        self.low = sorted(order[:int((left > REST ** 2).sum())].tolist())
        at = {q: nrow + j for j, q in enumerate(self.low)}
        self.terms += [(at[q], m) for q, m in self.terms if q in at]

    def _expand(self, monos, elements, char, inv):
        """Substitute x(u) into every monomial, keep the invariant ones and collect weights."""
        width = max(len(r) for r in inv)
        iu = np.zeros((self.nvars, width), np.int64)
        iw = np.zeros((self.nvars, width))
        for v, r in enumerate(inv):
            for j, (u, w) in enumerate(r):
                iu[v, j], iw[v, j] = u, w
        cu = np.zeros((self.nvars, len(elements)), np.int64)  # the same by character (one u each at most)
        cw = np.zeros((self.nvars, len(elements)))
        for v, r in enumerate(inv):
            for u, w in r:
                cu[v, char[u]], cw[v, char[u]] = u, w
        total = collections.Counter()
        by = collections.defaultdict(list)
        for k, m in monos:
            by[len(m)].append((k,) + tuple(m))
        base = self.nvars + 1
        for deg, rows in by.items():
            a = np.array(rows, np.int64)
            k, m = a[:, 0], a[:, 1:]
            # one monomial of each orbit, times the orbit's size: the others have the same invariant part
            images = np.stack([_key(np.sort(np.asarray(p)[m], axis=1), base) for p in elements])
            first = images[0] == images.min(axis=0)
            images = np.sort(images[:, first], axis=0)
            size = 1 + (images[1:] != images[:-1]).sum(axis=0)
            k, m = k[first], m[first]
            keys, weights = [], []
            for pick in itertools.product(range(width), repeat=max(deg - 1, 0)):
                w = size.astype(float)
                c = np.zeros(len(m), np.int64)
                u = np.empty_like(m)
                for d, j in enumerate(pick):
                    u[:, d] = iu[m[:, d], j]
                    w = w * iw[m[:, d], j]
                    c ^= char[u[:, d]]
                if deg:  # the last factor is the one with the product of the others' characters
                    u[:, -1] = cu[m[:, -1], c]
                    w = w * cw[m[:, -1], c]
                ok = w != 0
                u = np.sort(u[ok], axis=1)
                keys.append(_key(np.concatenate([k[ok, None], u], axis=1), base))
                weights.append(w[ok])
            key, at = np.unique(np.concatenate(keys), return_inverse=True)
            for q, w in zip(key.tolist(), np.bincount(at, weights=np.concatenate(weights)).tolist()):
                if w != 0.0:
                    mono = []
                    for _ in range(deg):
                        q, r = divmod(q, base)
                        mono.append(r)
                    total[(tuple(reversed(mono)), q)] = w
        rows = collections.defaultdict(list)
        for (mono, k), w in sorted(total.items()):
            rows[mono].append((k, w))
        # one slot per distinct combination, numbered in the order of its first coefficient
        slots = {r: q for q, r in enumerate(sorted(set(tuple(r) for r in rows.values())))}
        self.rows = sorted(slots, key=slots.get)
        self.terms = [(slots[tuple(r)], mono) for mono, r in rows.items()]


def _check_invariant(name, nvars, monos, perms):
    by = collections.defaultdict(list)
    for k, m in monos:
        by[len(m)].append((k,) + tuple(m))

    def canonical(a):
        a = a.copy()
        a[:, 1:] = np.sort(a[:, 1:], axis=1)
        return a[np.lexsort(a.T[::-1])]

    for rows in by.values():
        a = np.array(rows, np.int64)
        ref = canonical(a)
        for p in perms:
            b = a.copy()
            b[:, 1:] = np.asarray(p)[a[:, 1:]]
            if not np.array_equal(canonical(b), ref):
                raise ValueError("%s: an exchange of EXCHANGES is not a symmetry of the table" % name)


def emit_transform(fn, blocks):
    """In-place Walsh-Hadamard transform of every orbit (its own transpose)."""
    out = ["__device__ __forceinline__ void %s(double* v) {" % fn]
    for orbit in blocks:
        step = 1
        while step < len(orbit):
            for i in range(len(orbit)):
                if not i & step:
                    p, q = orbit[i], orbit[i + step]
                    out.append("    { const double a = v[%d], b = v[%d]; v[%d] = a + b; v[%d] = a - b; }" % (p, q, p, q))
            step *= 2
    out += ["}", ""]
    return "\n".join(out)


def emit_tables(name, sym, ncoef, transposed=False):
    """C arrays of T in compressed rows (b_q = sum a[k] w) and the slots with a second coefficient; with
    transposed the columns of T too."""
    rows = sym.rows
    out = ["// GENERATED by mbx_amd/gen/polygen.py from mbx_amd/tables/%s.tbl -- do not edit." % name,
           "// Coefficients of the symmetry-adapted polynomial from the fitted ones: b[q] = sum_i a[K[i]] W[i],",
           "// i in [Row[q], Row[q + 1]), rounded; b[NRow + j] is what rounding left of slot Low[j].", "#pragma once", ""]

    def arrays(tag, lists, cols):
        start = [0]
        for r in lists:
            start.append(start[-1] + len(r))
        flat = [t for r in lists for t in r]
        out.append("MBXG_SYM_SPACE const int kSym%sRow_%s[%d] = {" % (tag, name, len(start)))
        for i in range(0, len(start), 16):
            out.append("    " + ", ".join(str(v) for v in start[i:i + 16]) + ",")
        out.append("};")
        out.append("MBXG_SYM_SPACE const unsigned short kSym%sK_%s[%d] = {" % (tag, name, max(len(flat), 1)))
        for i in range(0, len(flat), 16):
            out.append("    " + ", ".join(str(k) for k, _ in flat[i:i + 16]) + ",")
        out.append("};")
        out.append("MBXG_SYM_SPACE const double kSym%sW_%s[%d] = {" % (tag, name, max(len(flat), 1)))
        for i in range(0, len(flat), 8):
            out.append("    " + ", ".join("%.17g" % w for _, w in flat[i:i + 8]) + ",")
        out.append("};")

    out.append("static constexpr int kNRow_%s = %d, kNLow_%s = %d, kNSlot_%s = %d;" % (
        name, len(rows), name, len(sym.low), name, len(rows) + len(sym.low)))
    arrays("", rows, ncoef)
    out.append("MBXG_SYM_SPACE const unsigned short kSymLow_%s[%d] = {%s};" % (
        name, max(len(sym.low), 1), ", ".join(str(q) for q in sym.low) or "0"))
    if transposed:
        cols = [[] for _ in range(ncoef)]
        for q, r in enumerate(rows):
            for k, w in r:
                cols[k].append((q, w))
        out.append("// the transpose: da[k] = sum_i db[TK[i]] TW[i]")
        arrays("T", cols, len(rows))
    return "\n".join(out) + "\n"
