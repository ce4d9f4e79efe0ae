"""The FP64 immersed boundary over markers at every edge: stencils that leave
the box in x and z (one or both axes folded), next to the first and last cells
that y allows, cells that no, one or many markers reach.  The
periodic step is the oracle's bit for bit; between walls a Newtonian step
differs by the transform's last bits only (1e-14)."""
import numpy as np
import pytest

from fortran8_amd import api, configs
from fortran8_amd.fields import Markers, State, interior, pad_periodic, ghosted_zeros, rel_l2, seeded_normal
from fortran8_amd.params import METHOD_IBM, default_params
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def case_of(nx, ny, nz, nl, walls):
    dx = 1.0 / 16
    p = default_params(nx=nx, ny=ny, nz=nz, lx=nx * dx, ly=ny * dx, lz=nz * dx, dt=1e-3, re=100.0, beta=1.0,
                       method=METHOD_IBM, walls_y=walls, body_force=(0.1, 0.02, 0.0))
    r = seeded_normal(nx + 31 * ny + 7 * nz, 3 * nx * ny * nz).reshape(3, nz, ny, nx)
    u = 0.2 * r
    u[0] += 1.0
    if walls:
        u[1][:, -1, :] = 0.0
    st = State(*[pad_periodic(a) for a in u], ghosted_zeros(nx, ny, nz),
               np.pad(np.broadcast_to(np.array([1.0, 0, 0, 1, 0, 1]), (nz, ny, nx, 6)),
                      ((1, 1), (1, 1), (1, 1), (0, 0)), mode="wrap").copy())
    # two "cylinders" of nl markers in every plane: along the x faces and
    # across the box, from the first row to the last that a marker may take
    t = np.linspace(0.0, 1.0, nl)
    x = np.stack([np.where(np.arange(nl) % 2 == 0, 0.5, nx - 0.5) + 0.3 * t * np.where(np.arange(nl) % 2 == 0, 1, -1),
                  0.5 + (nx - 1) * t])
    y = np.stack([1.5 + (ny - 3) * t, 1.5 + (ny - 3) * (1 - t) ** 2])
    x = np.broadcast_to(np.clip(x, 0.5, nx - 0.5) * dx, (nz, 2, nl))
    y = np.broadcast_to(y * dx, (nz, 2, nl))
    z = np.broadcast_to(((np.arange(nz) + 0.5) * dx)[:, None, None], (nz, 2, nl))
    uc = seeded_normal(5, 6 * nz * nl).reshape(3, nz, nl, 2) * 0.1
    m = Markers(2, nl, *[np.ascontiguousarray(np.swapaxes(a, 1, 2)) for a in (x, y, z)], *[a.copy() for a in uc])
    return configs.Case("edge_markers", p, st, markers=m)


@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape,nl", [((16, 16, 4), 7), ((4, 4, 4), 1), ((32, 8, 8), 70), ((4, 8, 16), 40)])
def test_edge_markers(shape, nl, walls):
    case = case_of(*shape, nl, walls)
    print("ibm case", shape, nl, "walls", walls, flush=True)
    o, g = po.load_case(case), api.load_case(case)
    o.step(2)
    g.step(2)
    so, sg = o.get_state(), g.get_state()
    fo, fg = np.stack(o.marker_forces()), np.stack(g.marker_forces())
    pairs = [(k, interior(getattr(sg, k)), interior(getattr(so, k))) for k in ("U", "V", "W", "P")]
    for name, a, b in pairs + [("F", fg, fo)]:
        assert np.isfinite(a).all(), name
        if walls:
            assert rel_l2(a, b) < 1e-14, (name, rel_l2(a, b))
        else:
            assert np.array_equal(a, b), (name, rel_l2(a, b))
    o.close()
    g.close()
