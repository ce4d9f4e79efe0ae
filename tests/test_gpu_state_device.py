"""The mixed state through device arrays against the same calls through the
host: any subset of outputs, arrays aligned to 8 bytes only, host memory as
source, and the histories, which a copy-out keeps (has_history = 1 or 2
continues with those of the last copy-out, also when steps ran in between).
Whole-number equality: both routes are conversions."""
import ctypes as C

import numpy as np
import pytest

from fortran8_amd import api, configs
from fortran8_amd.fields import interior, interior_c

pytestmark = pytest.mark.gpu
HIP = C.CDLL("libamdhip64.so.7")


class Planes:
    """U, V, W, P and C of n cells in device memory, `skew` doubles off its alignment"""

    def __init__(self, n, skew=0):
        self.base = C.c_void_p()
        assert HIP.hipMalloc(C.byref(self.base), C.c_size_t(8 * (10 * n + 8))) == 0
        self.n, self.at = n, [self.base.value + 8 * (skew + q * n) for q in range(5)]

    def read(self):
        out = np.empty((10, self.n))
        assert HIP.hipMemcpy(out.ctypes.data_as(C.c_void_p), C.c_void_p(self.at[0]), C.c_size_t(out.nbytes), 2) == 0
        return out

    def free(self):
        assert HIP.hipFree(self.base) == 0


def host(g):
    s = g.get_state()
    c = interior_c(s.C)
    return np.concatenate([np.stack([interior(a).ravel() for a in (s.U, s.V, s.W, s.P)]),
                           np.moveaxis(c.reshape(-1, 6), 1, 0)]), s.hist[:6]


@pytest.mark.parametrize("skew", [0, 1])
@pytest.mark.parametrize("walls", [0, 1])
def test_mixed_state_through_device_arrays(walls, skew):
    case = configs.channel_cylinder(nx=64, ny=32, nz=16, precision=1) if walls else configs.kolmogorov(n=16, precision=1)
    lib = api.lib()
    g = api.load_case(case)
    n = case.params.nx * case.params.ny * case.params.nz
    d = Planes(n, skew)
    g.step(2)
    assert lib.fp_get_state_device(g.h, *d.at, None) == 0
    state, hist = host(g)
    assert np.array_equal(d.read(), state)
    # a subset leaves the rest alone, and steps after a copy-out are as without
    g.step(1)
    assert lib.fp_get_state_device(g.h, None, d.at[1], None, None, None, None) == 0
    mixed = d.read()
    now, hist1 = host(g)
    assert np.array_equal(mixed[1], now[1]) and np.array_equal(np.delete(mixed, 1, 0), np.delete(state, 1, 0))
    h = api.load_case(case)
    h.step(3)
    assert all(np.array_equal(a, b) for a, b in zip(host(h), (now, hist1)))
    # back to the state of two steps with the histories of the last copy-out
    # (step 3's), once straight after it and once after more steps
    assert lib.fp_get_state_device(h.h, *d.at, None) == 0
    a = d.read()
    results = []
    for between in (0, 2):
        h.step(between)
        assert lib.fp_set_state_device(h.h, *d.at, 1 + (between > 0), None) == 0
        got, hh = host(h)          # (a copy-out too: the histories are again these)
        assert np.array_equal(got, a) and np.array_equal(hh, hist1)
        h.step(2)
        results.append(host(h))
        assert lib.fp_set_state_device(h.h, *d.at, 0, None) == 0
        h2 = api.load_case(case)
        assert lib.fp_set_state_device(h2.h, *d.at, 0, None) == 0
        h.step(2)
        h2.step(2)
        assert all(np.array_equal(x, y) for x, y in zip(host(h), host(h2)))
        h2.close()
        # the histories of step 3 for the next turn
        s3 = g.get_state()
        h.set_state(s3)
        assert lib.fp_get_state_device(h.h, *[None] * 5, None) == 0
    # a start from host memory takes copies
    s = a.copy()
    pinned = C.c_void_p()
    assert HIP.hipHostMalloc(C.byref(pinned), C.c_size_t(s.nbytes), 0) == 0
    C.memmove(pinned, s.ctypes.data, s.nbytes)
    assert lib.fp_set_state_device(h.h, *[pinned.value + 8 * q * n for q in range(5)], 0, None) == 0
    assert np.array_equal(host(h)[0], a)
    assert HIP.hipHostFree(pinned) == 0
    for x in (g, h):
        x.close()
    d.free()
    if not walls:   # the potential plays no part: both continuations are one
        assert all(np.array_equal(x, y) for x, y in zip(*results))
