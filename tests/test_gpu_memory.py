"""Device memory: what a step needs is allocated when the context is made."""
import ctypes as C

import pytest

from fortran8_amd import api, configs
from fortran8_amd.params import POISSON_SOR

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert api.lib().hipDeviceSynchronize() == 0
    assert api.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("case", [configs.channel_cylinder(), configs.kolmogorov(n=64),
                                  configs.channel_cylinder(nx=64, ny=32, nz=32, poisson_variant=POISSON_SOR)],
                         ids=["walls", "periodic", "sor"])
def test_steps_allocate_nothing(case):
    for _ in range(4):              # code objects and the runtime's buffers of its queues
        warm = api.load_case(case)
        warm.step(2)
        warm.close()
    g = api.load_case(case)
    before = free_bytes()
    g.step(2)
    assert free_bytes() == before
    g.close()


def test_a_mixed_context_holds_one_component_of_the_fp64_spectrum():
    """256^3: 264 B a cell of FP64 planes, 9 of selections and iteration counts,
    214 of the mixed step, 8 of the FP64 spectrum's one component; two more
    would be 16"""
    p = configs.kolmogorov(n=16, precision=1).params
    p.nx = p.ny = p.nz = 256
    api.FenepGPU(p).close()
    before = free_bytes()
    g = api.FenepGPU(p)
    used = (before - free_bytes()) / 256 ** 3
    g.close()
    assert 264 + 9 + 214 < used < 264 + 9 + 214 + 8 + 8
