"""The SOR sweeps on the tiles of 4 x 4 and 4 x 2 rows, which grids of 2048
and 4096 (y, z) lines and more take: x-lines of the fixed lengths and of others,
both boundary kinds.  FP64: the red-black iteration of numpy bit for bit.
FP32 (the mixed step): the sweeps that the FP64 step needs on its own, and its
velocity."""
import numpy as np
import pytest

from fortran8_amd import api
from fortran8_amd.fields import interior, rel_l2
from fortran8_amd.params import METHOD_FFT
from test_gpu_sor import case_of, red_black

pytestmark = pytest.mark.gpu

# 4 x 2: 2048 lines, or 256 points in x; 4 x 4: from 4096 lines on
TILES = [(16, 64, 32), (64, 64, 32), (128, 32, 64), (256, 64, 32), (4, 64, 64), (16, 64, 64), (32, 128, 32), (64, 64, 64),
         (128, 64, 64)]


@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", TILES)
def test_fp64_sweeps_on_larger_tiles(shape, walls):
    for itrmax in (1, 13):
        case = case_of(*shape, walls, itrmax=itrmax, eps=0.0)
        print("sor tile", shape, walls, itrmax, flush=True)
        g = api.load_case(case)
        g.step(1)
        phi, sweeps = red_black(case)
        assert g.diagnostics()["sor_itr"] == sweeps == itrmax
        assert np.array_equal(interior(g.get_phi()), phi), rel_l2(interior(g.get_phi()), phi)
        g.close()


# (512 points: FP32 alone, two trips of the tile's loads)
@pytest.mark.parametrize("walls", [0, 1])
@pytest.mark.parametrize("shape", TILES + [(256, 64, 64), (512, 64, 32)])
def test_mixed_sweeps_on_larger_tiles(shape, walls):
    print("mixed sor tile", shape, walls, flush=True)
    got = []
    for precision in (1, 0):
        case = case_of(*shape, walls, precision=precision, eps=1e-2)
        case.params.method = METHOD_FFT
        g = api.load_case(case)
        g.step(1)
        got.append((int(g.diagnostics()["sor_itr"]), g.get_state()))
        g.close()
    assert got[0][0] == got[1][0] > 0
    # the FP64 step ends its batch of ten: its velocity at the same sweep
    case.params.sor_itrmax = got[0][0]
    g = api.load_case(case)
    g.step(1)
    u = lambda st: np.stack([interior(st.U), interior(st.V), interior(st.W)])  # noqa: E731
    assert rel_l2(u(got[0][1]), u(g.get_state())) < 2e-6
    g.close()
