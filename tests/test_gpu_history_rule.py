"""The histories that fp_set_state_device takes with has_history = 1 and 2
(include/fenep_gpu.h): those of the last step on an FP64 context, those of the
last call that read the state out on a mixed one, where diagnostics and
statistics count as one."""
import ctypes as C

import numpy as np
import pytest

from fortran8_amd import api, configs
from test_gpu_state_device import Planes, host

pytestmark = pytest.mark.gpu


def read_out(g, call, d):
    if call == "get_state_device":
        assert api.lib().fp_get_state_device(g.h, *[None] * 5, None) == 0
    elif call == "diagnostics_static":
        from fortran8_amd.params import FpDiag
        assert api.lib().fp_diagnostics_static(g.h, C.byref(FpDiag())) == 0
    elif call is not None:
        getattr(g, call)()


@pytest.mark.parametrize("call", ["diagnostics", "diagnostics_static", "time_stats", "time_stats_map", "energy_spectrum",
                                  "energy_spectrum_z", "get_phi", "get_state"])
@pytest.mark.parametrize("precision", [0, 1])
def test_a_read_out_between_copy_out_and_set(precision, call):
    case = configs.kolmogorov(n=16, precision=precision)
    d = Planes(16 ** 3)
    results = {}
    for c in (None, call, "get_state_device"):
        g = api.load_case(case)
        g.step(2)
        assert api.lib().fp_get_state_device(g.h, *d.at, None) == 0
        g.step(2)
        read_out(g, c, d)
        g.step(1)
        assert api.lib().fp_set_state_device(g.h, *d.at, 2, None) == 0
        g.step(1)
        results[c] = host(g)
        g.close()
    d.free()
    same = lambda a, b: all(np.array_equal(x, y) for x, y in zip(results[a], results[b]))  # noqa: E731
    assert same(call, "get_state_device")
    # the mixed context's rule is visible: without the call it takes step 2's
    assert same(None, call) == (precision == 0)
