"""The intervals of the FP64 C+- selection (lowest and decide in
fortran8_amd/csrc/fp_select_f64.hip) on a float64 model: they hold the
reference's value (vieta_d, fenep.f90:425-444) of every candidate, and every
decision they make is the reference's (fenep.f90:186-221)."""
import os
import re

import numpy as np
import pytest

from test_select_certificate import vieta_ref
from test_select_certificate_f64 import FAMILIES, cells, reference

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fortran8_amd", "csrc", "fp_select_f64.hip")


def constants():
    s = open(SRC).read()
    psi = [float(x) for x in re.search(r"PSI\[11\] = \{([^}]*)\}", s).group(1).replace("\n", " ").split(",")]
    num = lambda name: float(re.search(name + r" = ([-+0-9.e]+)", s).group(1))  # noqa: E731
    lo, hi = re.search(r"r2 >= ([0-9.e+-]+) && r2 <= ([0-9.e+-]+)", s).groups()
    return np.array(psi), num("SEL_D3"), num("SEL_D0"), num("SEL_PSI_ERR"), float(lo), float(hi)


def exact_psi(s):
    return np.cos(2 * np.arcsin(np.clip(s / np.sqrt(2), -1, 1)) / 3 + 2 * np.pi / 3)


def lowest(a, rng):
    """(lambda, half-width, r); the hardware's reciprocal square roots are off by up to 2^-23"""
    psi, d3, d0, err, lo, hi = constants()
    rsq = lambda x: (1 + rng.uniform(-1, 1, x.shape) * 2.0 ** -23) / np.sqrt(x)  # noqa: E731
    with np.errstate(all="ignore"):
        m = ((a[0] + a[3]) + a[5]) * (1 / 3)
        b1, b2, b3 = a[0] - m, a[3] - m, a[5] - m
        o2 = a[1] * a[1] + (a[2] * a[2] + a[4] * a[4])
        r2 = (b1 * b1 + (b2 * b2 + b3 * b3)) * (1 / 6) + o2 * (1 / 3)
        det = b1 * (b2 * b3 - a[4] * a[4]) + (-a[1] * (a[1] * b3 - a[4] * a[2]) + a[2] * (a[1] * a[4] - b2 * a[2]))
        y = rsq(r2)
        ir = y + 0.5 * y * (1 - r2 * y * y)
        r = r2 * ir
        arg2 = det * (ir * ir * ir)
        s2 = 1 - 0.5 * arg2
        rho = abs(m) * ir + 2
        d = d3 * (rho * rho) * rho + d0
        w = np.fmax(s2, d)
        z = rsq(w)
        s = w * z
        s = s + 0.5 * s * (1 - s * z)
        ps = np.polynomial.polynomial.polyval(s, 2 * psi)
        ok = (abs(arg2) <= 2 - 4 * d) & (r2 >= lo) & (r2 <= hi)
        return r * ps + m, np.where(ok, r * (d * z + err), np.inf), r


def faces(cm, c, cp):
    return ([(c * 3.0) / 2.0 - cp / 2.0, cm / 2.0 + c / 2.0, (cm / 4.0 + c) - cp / 4.0],
            [c / 2.0 + cp / 2.0, -(cm / 2.0) + (c * 3.0) / 2.0, (-(cm / 4.0) + c) + cp / 4.0])


def decide(cm, c, cp, rng):
    """(option or -1, needed levels (3, n))"""
    lo, hi = [], []
    for p, q in zip(*faces(cm, c, cp)):
        (a, ea, _), (b, eb, _) = lowest(p, rng), lowest(q, rng)
        v, e = np.fmin(a, b), np.fmax(ea, eb)
        with np.errstate(all="ignore"):
            lo.append(v - e)
            hi.append(v + e)
    lo, hi = lo + [np.zeros_like(lo[0])], hi + [np.zeros_like(lo[0])]
    top = np.fmax.reduce(lo)
    can = np.array([~(h < top) for h in hi])
    return np.where(can.sum(0) == 1, can.argmax(0), -1), can[:3]


def test_polynomial():
    psi, _, _, err, _, _ = constants()
    t = np.linspace(0, np.sqrt(2), 400001)
    assert np.abs(np.polynomial.polynomial.polyval(t, psi) - exact_psi(t)).max() < 7.2e-11 and err > 2 * 7.2e-11


SIZES = [1e-160, 1e-52, 1e-44, 1e-30, 1e-3, 1.0, 1e30, 1e44, 1e52, 1e110]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("family", FAMILIES)
def test_intervals_hold_the_reference(family, size):
    rng = np.random.default_rng(FAMILIES.index(family) + 100 * SIZES.index(size))
    cm, c, cp = (a * size for a in cells(family, rng, 20000))
    worst = 0.0
    for a in sum(faces(cm, c, cp), []):
        v, e, _ = lowest(a, rng)
        ref = vieta_ref(a)
        ok = np.isfinite(e)
        assert np.all(abs(v - ref)[ok] <= e[ok]), (family, size)
        assert not np.any(np.isnan(ref[ok]) | (ref[ok] == -100.0))
        if ok.any():
            worst = max(worst, float((abs(v - ref)[ok] / e[ok]).max()))
    print(family, size, worst)


@pytest.mark.parametrize("size", [1e-52, 1.0, 1e44])
@pytest.mark.parametrize("family", FAMILIES)
def test_decisions_are_the_references(family, size):
    rng = np.random.default_rng(FAMILIES.index(family) + 7)
    cm, c, cp = (a * size for a in cells(family, rng, 60000))
    got, need = decide(cm, c, cp, rng)
    ref = reference(cm, c, cp)
    assert not np.any((got >= 0) & (got != ref))
    # a level that is not needed is never the answer
    sure = ref < 3
    assert np.all(np.take_along_axis(need, np.where(sure, ref, 0)[None], 0)[0][sure])


def test_equal_cells_have_two_distinct_levels():
    """the faces that the kernel leaves out where the three cells are the same"""
    c = cells("rough", np.random.default_rng(3), 1000)[1]
    left, right = faces(c, c, c)
    same = lambda a, b: np.array_equal(a.view(np.uint64), b.view(np.uint64))  # noqa: E731
    assert same(left[0], right[1]) and same(left[1], right[0])
