"""Captured batches after the Voronoi cells were replaced: the cells' arrays are
freed and allocated anew, and a batch captured before must not be replayed on
them unless every one of its pointers is the same."""
import numpy as np
import pytest

import openrbc_amd as orbc
from test_gpu_graphs import _sim, _states
from test_gpu_halo import _rbc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
def test_batches_after_new_cells(precision):
    s = _rbc(2)
    sims = [_sim(s, g, precision, seed=5, skin=0.1, volume_target=-1.0, volume_strength=0.2, freq_cleanup=20)
            for g in (1, 0)]
    for sim in sims:
        sim.minimize(20)
        sim.voronoi_init(0, 4)
        sim.run(37)
        c = np.asarray(sim.voronoi_get()[0]).reshape(-1, 3)
        # other sizes in between, so that arrays can change places
        for k in (len(c), len(c) // 2, len(c) - 3, len(c)):
            sim.voronoi_set_centroids(c[:k])
            sim.run(11)
    a, b = (_states(sim) for sim in sims)
    for sp in a:
        for k in a[sp]:
            assert np.array_equal(a[sp][k], b[sp][k]), (sp, k)
    assert sims[0].observables()["graph_replays"] > 0 and sims[1].observables()["graph_replays"] == 0
    for x, y in zip(sims[0].voronoi_get(), sims[1].voronoi_get()):
        assert np.array_equal(x, y)
    for sim in sims:
        sim.close()
