"""Fields read into arrays that overlap: the later field's numbers stand, in
page-locked memory as in ordinary one."""
import ctypes as C

import numpy as np
import pytest

import openrbc_amd as orbc
from test_gpu_readback import _Locked, _sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("locked", [False, True])
@pytest.mark.parametrize("shift", [0, 1, 30000])
def test_overlapping_arrays(shift, locked):
    with _sim(300, 200, 3, orbc.MIXED) as sim:
        mem = _Locked(sim.L)
        sim.run(2)
        want, m = sim.get_state(orbc.LIPID), 3 * sim.n[orbc.LIPID]
        buf = mem.array(m + 2 * shift) if locked else np.empty(m + 2 * shift)
        double = C.POINTER(C.c_double)
        ptr = [buf[k * shift:].ctypes.data_as(double) for k in range(3)]
        sim._check(sim.L.orbc_get_state(sim.h, orbc.LIPID, ptr[0], None, ptr[1], ptr[2]))
        for k, name in enumerate("xno"):
            a = buf[k * shift:k * shift + m] if k == 2 else buf[k * shift:(k + 1) * shift]
            assert np.array_equal(a, want[name].ravel()[:len(a)])
        mem.free()
