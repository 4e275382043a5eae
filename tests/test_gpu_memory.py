"""Device memory of a context: FP64 has no use for the FP32 mirrors (64 bytes a
particle in two buffers)."""
import ctypes as C

import pytest

import openrbc_amd as orbc
from openrbc_amd import systems

pytestmark = pytest.mark.gpu


def _free(L):
    a, b = C.c_size_t(), C.c_size_t()
    assert L.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def test_fp64_keeps_no_mirrors():
    s = systems.planar_patch(1000, 500, seed=1)
    n = len(s["lipid_x"])
    used = {}
    for precision in (orbc.MIXED, orbc.FP64):
        with orbc.Simulation(precision=precision) as sim:
            before = _free(sim.L)
            sim.set_state(orbc.LIPID, s["lipid_x"], s["lipid_n"], s["lipid_id"])
            sim.build_neighbors()
            used[precision] = (before - _free(sim.L)) / n
    # f, t, their second buffers and the scratch of energies are twice as wide in FP64
    # (72 bytes more a particle); the mirrors' 64 are not there.  Allocations come in
    # steps of at most 2 MiB, some 50 of them in each context: 2 bytes a particle each.
    extra = used[orbc.FP64] - used[orbc.MIXED]
    print(f"bytes a particle: mixed {used[orbc.MIXED]:.0f}, FP64 {used[orbc.FP64]:.0f}", flush=True)
    assert extra < 40
