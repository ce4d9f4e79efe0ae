"""The SOR sweeps on tiles (several sweeps a launch) over the grid shapes that
take different tiles, both boundary kinds, and iteration caps that are no
multiple of a launch's or a batch's sweeps.

From rest, without pressure and polymer, the explicit predictor is u* = dt F
exactly, so the right-hand side is known and a red-black iteration in numpy,
in the kernel's operation order, gives phi bit for bit.  The FP32 sweeps of
the mixed step are compared with the FP64 step's (same sweeps, velocity to
FP32)."""
import math

import numpy as np
import pytest

from fortran8_amd import api, configs
from fortran8_amd.fields import State, interior, ghosted_zeros, rel_l2, seeded_normal
from fortran8_amd.params import METHOD_EXPLICIT, METHOD_FFT, POISSON_SOR, default_params

pytestmark = pytest.mark.gpu


def case_of(nx, ny, nz, walls, precision=0, itrmax=10000, eps=1e-4):
    p = default_params(nx=nx, ny=ny, nz=nz, lx=nx / 16, ly=ny / 20, lz=nz / 24, dt=1e-3, re=100.0, beta=1.0,
                       method=METHOD_FFT if precision else METHOD_EXPLICIT, walls_y=walls, poisson_variant=POISSON_SOR,
                       precision=precision, sor_itrmax=itrmax, sor_eps=eps, sor_omega=1.6)
    z = ghosted_zeros(nx, ny, nz)
    st = State(z, z.copy(), z.copy(), z.copy(), np.zeros((nz + 2, ny + 2, nx + 2, 6)))
    f = seeded_normal(nx + 3 * ny + 7 * nz, 3 * nx * ny * nz).reshape(3, nz, ny, nx)
    return configs.Case("sor", p, st, force=tuple(f))


def red_black(case):
    """(phi, sweeps) in the kernel's order"""
    p = case.params
    dx, dy, dz = p.lx / p.nx, p.ly / p.ny, p.lz / p.nz
    u, v, w = (p.dt * f for f in case.force)
    below = np.roll(v, 1, 1)
    if p.walls_y:
        v = v.copy()
        v[:, -1] = 0.0
        below = np.concatenate([np.zeros_like(v[:, :1]), v[:, :-1]], 1)
    q = (((-np.roll(u, 1, 2) + u) / dx + (-below + v) / dy) + (-np.roll(w, 1, 0) + w) / dz) / p.dt
    bx, by, bz = 1.0 / (dx * dx), 1.0 / (dy * dy), 1.0 / (dz * dz)
    b0 = ((((bx + bx) + by) + by) + bz) + bz
    k, j, i = np.indices(q.shape)
    phi, done, er0 = np.zeros_like(q), 0, np.sum(q * q)
    while done < p.sor_itrmax:
        batch, met = min(10, p.sor_itrmax - done), 0
        for s in range(batch):
            er = 0.0
            for color in (0, 1):
                lo, hi = np.roll(phi, 1, 1), np.roll(phi, -1, 1)
                if p.walls_y:
                    lo, hi = np.concatenate([phi[:, :1], phi[:, :-1]], 1), np.concatenate([phi[:, 1:], phi[:, -1:]], 1)
                e = (((((bz * np.roll(phi, 1, 0) + by * lo) + bx * np.roll(phi, 1, 2)) - b0 * phi)
                      + bx * np.roll(phi, -1, 2)) + by * hi) + bz * np.roll(phi, -1, 0) - q
                e = np.where((i + j + k) % 2 == color, e, 0.0)
                phi = phi + (p.sor_omega * e) / b0
                er += np.sum(e * e)
            if not met and math.sqrt(er / er0) < p.sor_eps:
                met = s + 1
        done += met or batch
        if met:
            break
    return phi, done


SHAPES = [(4, 4, 4), (8, 4, 16), (16, 32, 8), (64, 8, 8), (64, 16, 32), (128, 16, 4), (256, 8, 8), (512, 4, 4), (1024, 4, 4)]


@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_fp64_sweeps_are_the_red_black_iteration(shape, walls):
    for itrmax, eps in ((10000, 1e-3), (13, 0.0), (10, 0.0), (1, 0.0)):
        case = case_of(*shape, walls, itrmax=itrmax, eps=eps)
        print("sor case", shape, walls, itrmax, flush=True)
        g = api.load_case(case)
        g.step(1)
        phi, sweeps = red_black(case)
        assert g.diagnostics()["sor_itr"] == sweeps
        assert np.array_equal(interior(g.get_phi()), phi), rel_l2(interior(g.get_phi()), phi)
        g.close()


def test_no_right_hand_side_takes_no_sweep():
    case = case_of(16, 8, 8, 0)
    case.force = tuple(np.zeros_like(f) for f in case.force)
    for precision in (0, 1):
        case.params.precision, case.params.method = precision, METHOD_FFT
        g = api.load_case(case)
        g.step(2)
        assert g.diagnostics()["sor_itr"] == 0 and not np.any(g.get_phi())
        g.close()


@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_sweeps_follow_the_fp64_ones(shape, walls):
    print("mixed sor case", shape, walls, flush=True)
    # the mixed step stops at the sweep that meets the test; the FP64 step, which
    # finishes its batch of ten, is held to as many by its cap
    got, itrmax = [], 10000
    for precision in (1, 0):
        case = case_of(*shape, walls, precision=precision, itrmax=itrmax, eps=1e-4)
        case.params.method = METHOD_FFT
        g = api.load_case(case)
        g.step(1)
        itrmax = int(g.diagnostics()["sor_itr"])
        got.append((itrmax, g.get_state()))
        g.close()
    assert got[0][0] > 0 and got[0][0] == got[1][0]
    u = lambda st: np.stack([interior(st.U), interior(st.V), interior(st.W)])  # noqa: E731
    assert rel_l2(u(got[0][1]), u(got[1][1])) < 2e-6
