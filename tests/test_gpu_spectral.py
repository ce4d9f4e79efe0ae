"""The FP64 spectral solves over the grid shapes that take different kernels.

A kx slab in LDS or separate y and z transforms, short and long lines, every
remainder of log2 n against the stages of a pass, one component or three in a
launch, and the line solves between walls.  The step of the Newtonian fluid
runs through all four solves; periodic results are the oracle's bit for bit,
walled ones to 1e-14 (no polymer is involved, so no selection can differ)."""
import numpy as np
import pytest

from fortran8_amd import api, configs
from fortran8_amd.fields import State, interior, pad_periodic, ghosted_zeros, rel_l2, seeded_normal
from fortran8_amd.params import METHOD_FFT, default_params
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def newtonian(nx, ny, nz, walls):
    p = default_params(nx=nx, ny=ny, nz=nz, lx=2.0, ly=1.5, lz=1.0, dt=1e-3, re=50.0, beta=1.0, method=METHOD_FFT,
                       walls_y=walls)
    u = seeded_normal(nx * 7 + ny * 3 + nz, 3 * nx * ny * nz).reshape(3, nz, ny, nx) * 0.01
    if walls:
        u[1][:, -1, :] = 0.0
    st = State(*[pad_periodic(a) for a in u], ghosted_zeros(nx, ny, nz), np.zeros((nz + 2, ny + 2, nx + 2, 6)))
    return configs.Case("spectral", p, st)


@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", [(4, 4, 4), (8, 4, 16), (16, 32, 8), (32, 16, 4), (64, 8, 32), (128, 64, 4), (4, 64, 128),
                                   (8, 128, 128), (16, 256, 64), (256, 8, 256), (4, 512, 32), (4, 16, 512), (512, 4, 8),
                                   (1024, 4, 4), (4, 1024, 8), (4, 8, 1024), (256, 128, 32)])
def test_newtonian_step_over_grid_shapes(shape, walls):
    case = newtonian(*shape, walls)
    print("spectral case", shape, "walls", walls, flush=True)
    o, g = po.load_case(case), api.load_case(case)
    o.step(2)
    g.step(2)
    so, sg = o.get_state(), g.get_state()
    for name in ("U", "V", "W", "P"):
        a, b = interior(getattr(sg, name)), interior(getattr(so, name))
        if walls:
            assert rel_l2(a, b) < 1e-14, (name, rel_l2(a, b))
        else:
            assert np.array_equal(a, b), (name, rel_l2(a, b))
    o.close()
    g.close()
