"""The FP64 conformation update and predictor over the grid shapes that take
different kernels, on a stretched, noisy conformation: the z-streamed
selection (nx 64, 128, 256), the per-cell one, short axes, both boundary
kinds.  Periodic steps are the oracle's bit for bit; between walls the ties of
the first rows are decided by the last bit of acos and the fields agree to
1e-14."""
import numpy as np
import pytest

from fortran8_amd import api, configs
from fortran8_amd.fields import State, interior, interior_c, pad_periodic, ghosted_zeros, rel_l2, seeded_normal
from fortran8_amd.params import METHOD_EXPLICIT, METHOD_FFT, default_params
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def stretched(nx, ny, nz, walls, method=METHOD_FFT):
    p = default_params(nx=nx, ny=ny, nz=nz, lx=nx / 16, ly=ny / 16, lz=nz / 16, dt=1e-3, re=100.0, beta=0.8, wi=1.5,
                       lp=9.0, method=method, walls_y=walls, body_force=(0.1, 0.02, 0.0))
    n = nx * ny * nz
    r = seeded_normal(nx + 31 * ny + 7 * nz, 12 * n).reshape(12, nz, ny, nx)
    u = 0.2 * r[:3]
    u[0] += 1.0
    if walls:
        u[1][:, -1, :] = 0.0
    f = 0.4 * r[3:].reshape(3, 3, nz, ny, nx) + np.eye(3)[:, :, None, None, None] * 1.5
    c = np.stack([np.einsum("kzyx,kzyx->zyx", f[a], f[b]) for a, b in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))], -1)
    st = State(*[pad_periodic(a) for a in u], ghosted_zeros(nx, ny, nz), np.pad(c, ((1, 1), (1, 1), (1, 1), (0, 0)), mode="wrap"))
    return configs.Case("stretched", p, st)


@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", [(4, 4, 4), (8, 16, 4), (64, 4, 8), (64, 16, 16), (128, 8, 4), (256, 4, 8), (512, 4, 4),
                                   (32, 32, 16), (64, 128, 64)])
def test_fenep_step_over_grid_shapes(shape, walls):
    case = stretched(*shape, walls)
    print("fenep case", shape, "walls", walls, flush=True)
    steps = 1 if shape[0] * shape[1] * shape[2] > 100000 else 3
    o, g = po.load_case(case), api.load_case(case)
    o.step(steps)
    g.step(steps)
    compare(o.get_state(), g.get_state(), walls)
    assert g.diagnostics()["newton_unconverged"] == 0
    o.close()
    g.close()


def test_explicit_method_step_is_the_oracles():
    case = stretched(16, 8, 32, 0, METHOD_EXPLICIT)
    o, g = po.load_case(case), api.load_case(case)
    o.step(3)
    g.step(3)
    compare(o.get_state(), g.get_state(), 0)


def compare(so, sg, walls):
    pairs = [(k, interior(getattr(sg, k)), interior(getattr(so, k))) for k in ("U", "V", "W", "P")]
    pairs += [("C", interior_c(sg.C), interior_c(so.C)), ("hist", sg.hist, so.hist)]
    for name, a, b in pairs:
        if walls:
            assert rel_l2(a, b) < 1e-14, (name, rel_l2(a, b))
        else:
            assert np.array_equal(a, b), (name, rel_l2(a, b))
