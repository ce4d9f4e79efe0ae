"""Infinities, NaN and zeros in the FP64 kernels that divide by a shared
divisor or choose face values by coefficients: a diverging run shows them in
the cells and values that the oracle's plain divisions and branches give, and a
zero keeps its sign."""
import numpy as np
import pytest

from fortran8_amd import api
from fortran8_amd.fields import interior, interior_c
from fortran8_amd.params import METHOD_EXPLICIT, POISSON_SOR
from oracle import pyoracle as po
from test_gpu_f64_fenep import stretched

pytestmark = pytest.mark.gpu


def planted(method, shape=(16, 16, 16), walls=0, **at):
    """the stretched case with values planted in fields: name=(value, component)"""
    case = stretched(*shape, walls, method)
    case.params.newton_itrmax = 20
    if method == METHOD_EXPLICIT:       # no sweeps: the new velocity is the predictor's
        case.params.poisson_variant = POISSON_SOR
        case.params.sor_itrmax = 0
    for name, (value, comp) in at.items():
        f = getattr(case.state, name)
        k, j, i = (s // 2 + 1 for s in shape[::-1])
        f[(k, j, i) if comp is None else (k, j, i, comp)] = value
    return case


def classes(a):
    return np.isnan(a) * 1 + np.isposinf(a) * 2 + np.isneginf(a) * 4


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("comp", [0, 1])
def test_conformation_update(value, comp):
    case = planted(1, C=(value, comp))
    o, g = po.load_case(case), api.load_case(case)
    o.step(1)
    g.step(1)
    a, b = interior_c(o.get_state().C), interior_c(g.get_state().C)
    assert np.array_equal(classes(a), classes(b))
    ok = np.isfinite(a)
    assert 0 < np.sum(~ok) < ok.size and np.array_equal(a[ok], b[ok])
    o.close()
    g.close()


@pytest.mark.parametrize("field", ["U", "V", "W", "P"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("shape", [(16, 16, 16), (64, 32, 32)])   # both predictor kernels
def test_predictor(shape, value, field):
    case = planted(METHOD_EXPLICIT, shape, **{field: (value, None)})
    o, g = po.load_case(case), api.load_case(case)
    o.step(1)
    g.step(1)
    s, t = o.get_state(), g.get_state()
    for f in "UVW":
        a, b = interior(getattr(s, f)), interior(getattr(t, f))
        assert np.array_equal(classes(a), classes(b)), f
        ok = np.isfinite(a)
        assert np.array_equal(a[ok], b[ok])
    o.close()
    g.close()


def test_zeros_keep_their_sign():
    case = planted(METHOD_EXPLICIT)
    case.params.body_force = (0.0, 0.0, 0.0)
    st = case.state
    for f in (st.U, st.V, st.W, st.P):
        f[:] = 0.0
    st.V[:] = -0.0
    st.C[:] = [1.0, 0.0, -0.0, 1.0, 0.0, 1.0]
    o, g = po.load_case(case), api.load_case(case)
    o.step(1)
    g.step(1)
    s, t = o.get_state(), g.get_state()
    for f in "UVW":
        a, b = interior(getattr(s, f)), interior(getattr(t, f))
        assert np.array_equal(a, b) and np.array_equal(np.signbit(a), np.signbit(b)), f
    assert np.array_equal(np.signbit(s.hist), np.signbit(t.hist))
    o.close()
    g.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_divergence_of_an_infinite_velocity(precision):
    case = planted(1, U=(np.inf, None))
    case.params.precision = precision
    g = api.load_case(case)
    d = g.diagnostics()
    assert d["div_max"] == np.inf and d["nan_flag"] == 0
    assert g.time_stats()[6] == np.inf      # the dissipation: |S|^2
    g.close()


def test_sor_sweep_of_an_infinite_right_hand_side():
    """one red-black sweep from zero"""
    case = planted(METHOD_EXPLICIT, P=(np.inf, None))
    g = api.load_case(case)
    g.step(1)                                 # no sweep: u* itself
    s = g.get_state()
    g.close()
    case.params.sor_itrmax = 1
    g = api.load_case(case)
    g.step(1)
    phi = interior(g.get_phi())
    g.close()
    p, h = case.params, case.params.lx / case.params.nx
    om, b = 2.0 / (1.0 + np.sin(np.pi * h)), 1.0 / (h * h)
    u, v, w = (interior(a) for a in (s.U, s.V, s.W))
    with np.errstate(all="ignore"):
        q = (((-np.roll(u, 1, 2) + u) / h + (-np.roll(v, 1, 1) + v) / h) + (-np.roll(w, 1, 0) + w) / h) / p.dt
        want = np.zeros_like(q)
        colour = np.indices(q.shape).sum(0) % 2
        for c in (0, 1):
            at = lambda o, ax: np.roll(want, -o, ax)  # noqa: E731
            e = (((((b * at(-1, 0) + b * at(-1, 1)) + b * at(-1, 2)) - (6.0 * b) * want) + b * at(1, 2)) + b * at(1, 1)) \
                + b * at(1, 0) - q
            want = np.where(colour == c, want + (om * e) / (6.0 * b), want)
    assert np.isinf(want).any() and np.isnan(want).any()
    assert np.array_equal(classes(phi), classes(want))
