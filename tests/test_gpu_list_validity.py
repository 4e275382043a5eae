"""After a run the neighbour list serves the state that the run left: the last
step's own skin check stands in for a pass over the positions.  The forces of
the list at hand must be those of a list built anew, after every run length up
to a list's life and past it, and the counts must be those of the observables."""
import ctypes as C

import numpy as np
import pytest

import openrbc_amd as orbc
from openrbc_amd import systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thermostat", [orbc.RUN_LANGEVIN, orbc.RUN_NOSE_HOOVER])
@pytest.mark.parametrize("skin", [0.02, 0.1])
def test_list_at_hand_after_a_run_is_valid(skin, thermostat):
    s = systems.planar_patch(20, 20, seed=2)
    x, n = s["lipid_x"], s["lipid_n"]
    v = np.random.default_rng(1).normal(0, 0.4, x.shape)
    rebuilt = 0
    with orbc.Simulation(precision=orbc.FP64, seed=4, skin=skin, thermostat=thermostat) as sim:
        sim.set_state(orbc.LIPID, x, n, s["lipid_id"], v=v)
        for steps in (1, 1, 2, 3, 0, 1, 5, 1, 1):
            before = sim.observables()["rebuilds"]
            sim.run(steps)
            rebuilt += sim.observables()["rebuilds"] - before
            nl, npr = C.c_longlong(), C.c_longlong()
            sim._check(sim.L.orbc_get_counts(sim.h, C.byref(nl), C.byref(npr)))
            assert (nl.value, npr.value) == (len(x), 0)
            now = sim.get_state(orbc.LIPID)
            with orbc.Simulation(precision=orbc.FP64, skin=skin) as ref:
                ref.set_state(orbc.LIPID, now["x"], now["n"], s["lipid_id"])
                f, fr = [], []
                for one, out in ((sim, f), (ref, fr)):
                    # Nose-Hoover keeps its forces for the next first half: read, then put back
                    kept = one.get_forces(orbc.LIPID) if one is sim else None
                    one.compute_pairwise(zero_first=True)
                    out.extend(one.get_forces(orbc.LIPID))
                    if kept is not None:
                        one.set_forces(orbc.LIPID, *kept)
            for a, b in zip(f, fr):
                # same pairs, summed in another order: a few hundred roundings of terms below 1e3
                assert np.abs(a - b).max() < 1e-10
    assert rebuilt >= 2
