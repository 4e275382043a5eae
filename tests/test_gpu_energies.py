"""Per-particle energies and virials stay with their particles: through re-sorts of
the store, runs that rebuild, and the removal of lipids."""
import ctypes as C

import numpy as np
import pytest

import openrbc_amd as orbc
from _systems import patch, split

pytestmark = pytest.mark.gpu
SPECIES = (orbc.LIPID, orbc.PROTEIN)


def _sim(precision, thermostat=orbc.RUN_LANGEVIN, skin=0.05):
    s = patch(18, 14, seed=4)
    lip, prot = split(s)
    sim = orbc.Simulation(precision=precision, seed=2, skin=skin, thermostat=thermostat, freq_cleanup=0)
    sim.set_state(orbc.LIPID, s["x"][lip], s["n"][lip], s["id"][lip], v=s["v"][lip])
    sim.set_state(orbc.PROTEIN, s["x"][prot], s["n"][prot], s["id"][prot], v=s["v"][prot], type=s["type"][prot])
    bt, bi, bj = s["bonds"]
    sim.set_bonds(bt, s["id"][bi], s["id"][bj])
    return sim, s, (lip, prot)


def _ew(sim):
    return [a for sp in SPECIES for a in sim.get_forces(sp, energy=True)[2:]]


@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
def test_energies_travel_with_the_store(precision):
    """What an evaluation left is what is read after the particles changed places in
    the store (mirrored positions reverse its order) and after a run that rebuilds."""
    sim, s, which = _sim(precision)
    sim.compute_pairwise(zero_first=True, energy=True)
    sim.compute_bonded(energy=True)
    want = _ew(sim)
    assert all(len(np.unique(a)) > len(a) // 2 for a in want)
    for sp, k in zip(SPECIES, which):
        sim.set_state(sp, s["x"][k] * [-1.0, -1.0, 1.0], s["n"][k], s["id"][k], v=s["v"][k],
                      type=s["type"][k] if sp == orbc.PROTEIN else None)
    sim.build_neighbors()
    for a, b in zip(want, _ew(sim)):
        assert np.array_equal(a, b)
    before = sim.observables()["rebuilds"]
    want = _ew(sim)                     # of the observables, as of the mirrored state
    sim._check(sim.L.orbc_run(sim.h, 30))
    for a, b in zip(want, _ew(sim)):
        assert np.array_equal(a, b)
    assert sim.observables()["rebuilds"] > before
    sim.close()


@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
def test_energies_of_the_lipids_that_stay(precision):
    sim, _, _ = _sim(precision)
    sim.voronoi_init(0, 4)
    sim.compute_pairwise(zero_first=True, energy=True)
    want, x = _ew(sim), sim.get_state(orbc.LIPID)["x"]
    gone = C.c_longlong()
    sim._check(sim.L.orbc_delete_stray_lipids(sim.h, 1.2, C.byref(gone)))
    assert 0 < gone.value < len(x)
    sim.n[orbc.LIPID] -= gone.value
    left = {tuple(r) for r in sim.get_state(orbc.LIPID)["x"]}
    keep = np.array([tuple(r) in left for r in x])
    assert keep.sum() == len(left) == len(x) - gone.value
    for a, b, k in zip(want, _ew(sim), (keep, keep, slice(None), slice(None))):
        assert np.array_equal(a[k], b)
    sim.close()


@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
@pytest.mark.parametrize("thermostat", [orbc.RUN_LANGEVIN, orbc.RUN_NOSE_HOOVER])
def test_energies_after_a_run(thermostat, precision):
    """A run leaves the energies and virials of its last state, those that the
    observables sum up, and the forces as it had them."""
    sim, _, _ = _sim(precision, thermostat)
    for steps in (0, 1, 25):
        sim.run(steps)
        got, forces = _ew(sim), [sim.get_forces(sp)[0] for sp in SPECIES]
        assert any(f.any() for f in forces) == (thermostat == orbc.RUN_NOSE_HOOVER)
        obs = sim.observables()
        for name, a in (("potential", np.r_[got[0], got[2]]), ("virial", np.r_[got[1], got[3]])):
            assert abs(obs[name] - a.sum()) <= 1e-13 * np.abs(a).sum()      # some 300 terms in another order
        for a, b in zip(got, _ew(sim)):
            assert np.array_equal(a, b)
        for f, sp in zip(forces, SPECIES):
            assert np.array_equal(f, sim.get_forces(sp)[0])
    sim.close()


def test_energies_after_cleanup_and_restart(tmp_path):
    sim, _, _ = _sim(orbc.FP64)
    sim.voronoi_init(0, 4)
    assert sim.delete_stray_lipids(1.2) > 0
    got = _ew(sim)
    assert all(a.any() for a in got)
    sim.save_restart(str(tmp_path / "r"))
    sim.observables()
    for a, b in zip(got, _ew(sim)):
        assert np.array_equal(a, b)
    sim.load_restart(str(tmp_path / "r"))
    for a, b in zip(got, _ew(sim)):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()      # same pairs, in the order of a new list
    sim.close()
