"""The FP64 step from states that leave much of the C+- selection to the
formula in FP64: cells equal or nearly equal along axes, isotropic ones, sizes
outside the intervals' range, on every instance of the kernel.  Ties are
decided by the last bit of acos and cos, between candidates equal to rounding:
the conformation agrees with the oracle's to 1e-14, as in test_gpu_f64_fenep."""
import numpy as np
import pytest

from fortran8_amd import api
from fortran8_amd.fields import interior_c, rel_l2
from oracle import pyoracle as po
from test_gpu_f64_fenep import stretched

pytestmark = pytest.mark.gpu


def state(kind, c, rng):
    """the interior conformation (nz, ny, nx, 6) of a state"""
    eye = np.broadcast_to(np.array([1.0, 0, 0, 1, 0, 1]), c.shape).copy()
    if kind == "at rest":
        return eye
    if kind.startswith("noise"):         # 1e-4: a few pairs a block
        return eye + float(kind.split()[1]) * rng.standard_normal(c.shape)
    if kind == "small":
        return 1e-60 * c
    c = np.broadcast_to(c[:1], c.shape).copy()
    if kind == "uniform in y and z":
        c = np.broadcast_to(c[:, :1], c.shape).copy()
    if kind == "half uniform":           # lists of every length from block to block
        c[c.shape[0] // 2:] *= 1 + 1e-3 * rng.random((c.shape[0] - c.shape[0] // 2,) + c.shape[1:])
    return c


KINDS = ["at rest", "noise 1e-15", "noise 1e-4", "small", "uniform in z", "uniform in y and z", "half uniform"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", [(4, 4, 4), (8, 4, 4), (16, 32, 8), (64, 16, 8), (256, 4, 4), (512, 4, 4), (128, 128, 64),
                                   (256, 128, 64)])   # blocks of one plane, then of two and of four
def test_conformation_where_candidates_tie(shape, walls, kind):
    case = stretched(*shape, walls)
    case.params.newton_itrmax = 30
    rng = np.random.default_rng(KINDS.index(kind))
    case.state.C[1:-1, 1:-1, 1:-1] = state(kind, interior_c(case.state.C).copy(), rng)
    case.state.C[:] = np.pad(interior_c(case.state.C), ((1, 1), (1, 1), (1, 1), (0, 0)), mode="wrap")
    print("selection", shape, walls, kind, flush=True)
    o, g = po.load_case(case), api.load_case(case)
    o.step(1)
    g.step(1)
    assert rel_l2(interior_c(g.get_state().C), interior_c(o.get_state().C)) < 1e-14
    o.close()
    g.close()
