"""Which arrays the GPU writes itself when state is read: those that lie whole in
one page-locked allocation (nothing is read or written here, addresses are asked)."""
import ctypes as C

import numpy as np
import pytest

import openrbc_amd as orbc
from test_gpu_readback import _Locked

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 600, 100003])
def test_only_whole_ranges_in_locked_memory(m):
    with orbc.Simulation() as sim:
        ask, mem = sim.L.orbc_test_reads_direct, _Locked(sim.L)
        ask.argtypes, ask.restype = [C.c_void_p, C.c_size_t], C.c_int
        a, b = mem.array(m), np.empty(m)
        p = a.ctypes.data
        assert ask(p, 8 * m) and ask(p, 8)
        assert ask(p + 8 * (m - 1), 8)
        assert not ask(p, 8 * m + 1) and not ask(p + 8, 8 * m) and not ask(p + 8 * (m - 1), 16)
        assert not ask(b.ctypes.data, 8 * m)
        mem.free()
        assert not ask(p, 8 * m)
