"""The mixed Helmholtz solve by 1 to 4 fixed-point sweeps in one kernel, over
tiles, halos that wrap, and both boundary kinds, against a launch per sweep
(5 sweeps).  With rho = eps lambda_max = 1e-3 here, S sweeps leave rho^(S+1)
of the increment d = u* - u: 1e-6 |d| for one sweep and nothing FP32 can hold
for more.  |d| / |u| is below 0.1 here, and each side rounds u to FP32 once
(2^-24) and d a few times: 3e-7 for every S."""
import numpy as np
import pytest

from fortran8_amd import api, configs
from fortran8_amd.fields import State, interior, pad_periodic, ghosted_zeros, rel_l2, seeded_normal
from fortran8_amd.params import METHOD_FFT, default_params

pytestmark = pytest.mark.gpu


def step(shape, walls, sweeps):
    nx, ny, nz = shape
    dx, dt, re = 1.0 / 16, 1e-3, 100.0
    re = 0.5 * dt * 12.0 / dx ** 2 / 1e-3          # rho = dt/(2 Re) 12/dx^2
    p = default_params(nx=nx, ny=ny, nz=nz, lx=nx * dx, ly=ny * dx, lz=nz * dx, dt=dt, re=re, beta=1.0,
                       method=METHOD_FFT, walls_y=walls, precision=1, helm_sweeps=sweeps, body_force=(0.1, 0.02, 0.0))
    u = 0.2 * seeded_normal(nx + 31 * ny + 7 * nz, 3 * nx * ny * nz).reshape(3, nz, ny, nx)
    u[0] += 1.0
    if walls:
        u[1][:, -1, :] = 0.0
    c = np.broadcast_to(np.array([1.0, 0, 0, 1, 0, 1]), (nz + 2, ny + 2, nx + 2, 6)).copy()
    st = State(*[pad_periodic(a) for a in u], ghosted_zeros(nx, ny, nz), c)
    g = api.load_case(configs.Case("sweeps", p, st))
    g.step(1)
    s = g.get_state()
    g.close()
    return [interior(a) for a in (s.U, s.V, s.W)]


@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", [(4, 4, 4), (8, 16, 4), (64, 8, 32), (128, 32, 8), (32, 64, 64), (256, 128, 32)])
def test_fused_sweeps(shape, walls):
    print("sweeps case", shape, "walls", walls, flush=True)
    want = step(shape, walls, 5)
    for sweeps in (1, 2, 3, 4):
        for a, b in zip(step(shape, walls, sweeps), want):
            assert rel_l2(a, b) < 3e-7, (sweeps, rel_l2(a, b))
