"""The mixed step's y and z transforms over every line length, in registers (16
to 256 points) and in the LDS (the others), against the FP64 step: Poisson and,
with the spectral Helmholtz solve, the other symbols; between walls the boxes
whose kx slab does not fit the LDS as well.  One step of noise of 0.2 on a
stream of 1: the FP32 transforms are good to about 2^-24 sqrt(log2 N) = 2.5e-7
of what they solve for, which is below |u|, and u is rounded to FP32 once: 1e-6."""
import numpy as np
import pytest

from fortran8_amd import api, configs
from fortran8_amd.fields import State, interior, pad_periodic, ghosted_zeros, rel_l2, seeded_normal
from fortran8_amd.params import METHOD_FFT, default_params

pytestmark = pytest.mark.gpu


def velocities(shape, walls, precision, sweeps):
    nx, ny, nz = shape
    dx = 1.0 / 16
    p = default_params(nx=nx, ny=ny, nz=nz, lx=nx * dx, ly=ny * dx, lz=nz * dx, dt=1e-3, re=100.0, beta=1.0,
                       method=METHOD_FFT, walls_y=walls, precision=precision, helm_sweeps=sweeps,
                       body_force=(0.1, 0.02, 0.0))
    u = 0.2 * seeded_normal(nx + 31 * ny + 7 * nz, 3 * nx * ny * nz).reshape(3, nz, ny, nx)
    u[0] += 1.0
    if walls:
        u[1][:, -1, :] = 0.0
    c = np.broadcast_to(np.array([1.0, 0, 0, 1, 0, 1]), (nz + 2, ny + 2, nx + 2, 6)).copy()
    g = api.load_case(configs.Case("lines", p, State(*[pad_periodic(a) for a in u], ghosted_zeros(nx, ny, nz), c)))
    g.step(1)
    s = g.get_state()
    g.close()
    return np.stack([interior(a) for a in (s.U, s.V, s.W)])


@pytest.mark.parametrize("sweeps", [0, -1])
@pytest.mark.parametrize("shape,walls", [((4, 4, 8), 0), ((8, 16, 4), 0), ((4, 32, 16), 0), ((32, 64, 32), 0),
                                         ((16, 128, 64), 0), ((4, 256, 128), 0), ((8, 8, 256), 0), ((4, 512, 16), 0),
                                         ((4, 16, 1024), 0), ((64, 64, 64), 0), ((8, 128, 256), 1), ((4, 512, 64), 1),
                                         ((16, 32, 16), 1), ((4, 256, 128), 1), ((4, 1024, 32), 1)])
def test_step_over_line_lengths(shape, walls, sweeps):
    print("lines case", shape, "walls", walls, "sweeps", sweeps, flush=True)
    a, b = velocities(shape, walls, 1, sweeps), velocities(shape, walls, 0, 0)
    assert rel_l2(a, b) < 1e-6, rel_l2(a, b)
