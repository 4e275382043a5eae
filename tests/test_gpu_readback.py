"""State and forces read into page-locked arrays (one kernel that writes them)
equal those read into ordinary ones (staged copies), number for number: sizes
around a block, arrays that start off a 16-byte boundary or are only partly
page-locked, both precisions and species."""
import ctypes as C

import numpy as np
import pytest

import openrbc_amd as orbc
from openrbc_amd import systems

pytestmark = pytest.mark.gpu


def _sim(nx, ny, proteins, precision):
    s = systems.planar_patch(nx, ny, seed=3)
    rng = np.random.default_rng(nx)
    x, n = s["lipid_x"], s["lipid_n"]
    sim = orbc.Simulation(precision=precision, seed=9)
    sim.set_state(orbc.LIPID, x, n, s["lipid_id"], v=rng.normal(0, 0.3, x.shape))
    px = np.stack([np.arange(proteins) * 4.0, np.zeros(proteins), np.full(proteins, -6.0)], 1)
    pn = np.tile([0.0, 0.0, 1.0], (proteins, 1))
    sim.set_state(orbc.PROTEIN, px, pn, np.arange(proteins, dtype=np.uint32) + s["lipid_id"].max() + 1,
                  type=np.full(proteins, 5, np.int32))
    return sim


class _Locked:
    """Page-locked memory of the HIP runtime the library uses."""

    def __init__(self, L):
        self.L, self.ptrs = L, []
        L.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
        L.hipHostFree.argtypes = [C.c_void_p]

    def array(self, m):
        p = C.c_void_p()
        assert self.L.hipHostMalloc(C.byref(p), 8 * m, 0) == 0
        self.ptrs.append(p)
        return np.frombuffer((C.c_double * m).from_address(p.value), np.float64)

    def free(self):
        for p in self.ptrs:
            self.L.hipHostFree(p)


def _array(m, width, locked, offset):
    a = locked.array(m * width + offset) if locked else np.empty(m * width + offset)
    a[:] = -7.0
    return a[offset:]


def _read(sim, entry, species, widths, locked, offset):
    m = sim.n[species]
    out = [_array(m, w, p, offset) for w, p in zip(widths, locked)]
    sim._check(entry(sim.h, species, *[a.ctypes.data_as(C.POINTER(C.c_double)) for a in out]))
    return out


@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
@pytest.mark.parametrize("nx,ny,proteins", [(5, 4, 1), (16, 16, 3), (257, 10, 300)])
def test_page_locked_arrays_hold_the_same_numbers(nx, ny, proteins, precision):
    with _sim(nx, ny, proteins, precision) as sim:
        locked = _Locked(sim.L)
        sim.run(3)
        sim.compute_pairwise(zero_first=True, energy=True)
        for entry, widths in ((sim.L.orbc_get_state, (3, 3, 3, 3)), (sim.L.orbc_get_forces, (3, 3, 1, 1))):
            for species in (orbc.LIPID, orbc.PROTEIN):
                want = _read(sim, entry, species, widths, (None,) * 4, 0)
                assert all(np.isfinite(a).all() for a in want)
                for where, offset in (((locked,) * 4, 0), ((locked,) * 4, 1), ((locked, None, locked, None), 3)):
                    got = _read(sim, entry, species, widths, where, offset)
                    for a, b in zip(want, got):
                        assert np.array_equal(a, b)
        locked.free()
