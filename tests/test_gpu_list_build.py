"""The neighbour list against lists made without it: cells whose 27 hold more than
the 256 candidates a wave has in registers, rows past the 48 entries collected in
LDS and past the rows allocated at first, far-reaching proteins among them, the
Voronoi stencil, and the sizes at which a wave takes 8, 16 or 64 particles.  Sums
over cells up to eight rounds, positions and directors, and the partition where a
position is not a number."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

import openrbc_amd as orbc
from openrbc_amd import systems
from test_gpu_dispatch import _lipids, _nearest
from test_gpu_halo import _run, _same, _with_blob
from test_gpu_parity import id_pairs

pytestmark = pytest.mark.gpu
SKIN = 0.4


def _cube(m, a, proteins, seed=7):
    rng = np.random.default_rng(seed)
    g = np.arange(m) * a
    x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) + rng.normal(0, 0.05 * a, (m ** 3, 3))
    n = rng.normal(size=x.shape)
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    t = rng.choice(6, len(x), p=[0.5] + [0.1] * 5) if proteins else np.zeros(len(x))
    return dict(x=x, n=n, type=t.astype(np.int32), id=rng.permutation(len(x)).astype(np.uint32) + 5)


def _sim(s, precision, **kw):
    sim = orbc.Simulation(precision=precision, skin=SKIN, **kw)
    lip, prot = (np.flatnonzero(k) for k in (s["type"] == 0, s["type"] != 0))
    sim.set_state(orbc.LIPID, s["x"][lip], s["n"][lip], s["id"][lip])
    sim.set_state(orbc.PROTEIN, s["x"][prot], s["n"][prot], s["id"][prot], type=s["type"][prot])
    return sim, lip, prot


def _entries(s, ff, reach):
    """Directed pairs within the list's cutoffs, moved by `reach`."""
    rc = np.maximum(ff["cut_poly"], np.sqrt(ff["cut2_lj"]))
    cut2 = np.where(rc > 0, (rc + SKIN + 1e-4 + reach) ** 2, -1.0)
    x, t, total, longest = s["x"], s["type"], 0, 0
    for i in range(0, len(x), 256):
        d = x[i:i + 256, None] - x[None]
        rows = ((d * d).sum(2) < cut2[t[i:i + 256, None], t[None]]).sum(1) - (rc[t[i:i + 256], t[i:i + 256]] > 0)
        total, longest = total + rows.sum(), max(longest, rows.max())
    return total, longest


# rows of some 110, 500 and 100 entries; 48 are collected in LDS and allocated at first
@pytest.mark.parametrize("precision", [orbc.FP64, orbc.MIXED])
@pytest.mark.parametrize("m,a,proteins", [(16, 1.0, False), (13, 0.6, False), (16, 1.0, True), (13, 0.6, True)])
def test_dense_cells(m, a, proteins, precision, oracle):
    s = _cube(m, a, proteins)
    sim, _, _ = _sim(s, precision)
    got, obs = sim.pairs(), sim.observables()
    if precision == orbc.FP64:
        want = oracle.pairs_brute(s["x"], s["type"])
    else:
        want = oracle.pairs_mixed(s["x"], s["type"], obs["anchor_h"])
    assert np.array_equal(got, id_pairs(s, want))
    # the list test is in FP32 (offsets in a cell, rounding below 1e-6 each)
    ff = oracle.ff()
    low, longest = _entries(s, ff, -4e-6)
    high, _ = _entries(s, ff, 4e-6)
    assert longest > 64 and low <= obs["pairs"] <= high
    sim.close()


@pytest.mark.parametrize("m,a", [(16, 1.0), (20, 0.75)])
def test_dense_cells_stencil(m, a, oracle):
    s = _cube(m, a, True)
    sim, lip, prot = _sim(s, orbc.FP64, neighbor_mode=orbc.NEIGHBOR_VORONOI)
    sim.voronoi_init(12, 3)
    c, al, ap = sim.voronoi_get()
    aff = np.zeros(len(s["x"]), np.int32)
    aff[lip], aff[prot] = al, ap
    c = np.asarray(c, np.float32).reshape(-1, 3)
    want = oracle.pairs_voronoi(s["x"], s["type"], aff, c)
    assert 0 < len(want) < len(oracle.pairs_brute(s["x"], s["type"]))
    assert np.array_equal(sim.pairs(), id_pairs(s, want))
    sim.close()


# 8 particles a wave below 131072, 16 below 524288, then 64
@pytest.mark.parametrize("n", [131071, 131072, 524287, 524288])
def test_particles_of_a_wave(n):
    nx = int(np.ceil(np.sqrt(n)))
    s = systems.planar_patch(nx, -(-n // nx), seed=5)
    x = s["lipid_x"][:n]
    sim = _lipids(x, s["lipid_n"][:n], v=False, precision=orbc.FP64, skin=SKIN)
    tree = cKDTree(x)
    want = np.sort(tree.query_pairs(2.6, output_type="ndarray"), axis=1)
    assert np.array_equal(sim.pairs(), want[np.lexsort((want[:, 1], want[:, 0]))])
    low, high = (tree.count_neighbors(tree, 2.6 + SKIN + 1e-4 + d) - n for d in (-4e-6, 4e-6))
    assert low <= sim.observables()["pairs"] <= high
    sim.close()


# more than 512 blocks: two threads share a row of the halo build
@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
def test_overflowing_halos_of_many_blocks(precision):
    p = systems.planar_patch(256, 512, seed=5)
    n = len(p["lipid_x"])
    s = dict(x=p["lipid_x"], n=p["lipid_n"], v=np.zeros((n, 3)), o=np.zeros((n, 3)), type=np.zeros(n, np.int32),
             id=p["lipid_id"], bonds=(np.zeros(0, np.int32),) * 3)
    s = _with_blob(s, offset=(20.0, 20.0, 40.0))
    on, obs = _run(s, 1, 4, minimize=20, precision=precision, seed=4, skin=0.2)
    off, _ = _run(s, 0, 4, minimize=20, precision=precision, seed=4, skin=0.2)
    _same(on, off)
    assert 512 < obs["halo_blocks"] and 0 < obs["halo_overflow"] < 100


# blocks of 256 lipids: one round below 1800, two below 3600, four below 7200, then eight
@pytest.mark.parametrize("blocks", [1, 1801, 3601, 7199, 7201])
def test_cell_sums_of_positions_and_directors(blocks):
    n = blocks * 256 - 3
    nx = int(np.ceil(np.sqrt(n)))
    s = systems.planar_patch(nx, -(-n // nx), tilt=0.3, seed=5)
    x, nrm = s["lipid_x"][:n], s["lipid_n"][:n]
    sim = _lipids(x, nrm, v=False, precision=orbc.FP64, skin=SKIN)
    sim.voronoi_init(0, 0)
    _, aff, _ = sim.voronoi_get()

    def sums(a, k):
        return np.stack([np.bincount(aff, a[:, d], k) for d in range(3)], 1)

    # the push is the cell's normal times a number; the first call adds all sums up with
    # atomics, the second stores those of the cells that a block holds whole
    for calls in (1, 2):
        vol = sim.constrain_volume(1.0, 0.5)
        f = sim.get_forces(orbc.LIPID)[0] / (calls * 0.5 * (1.0 - vol))
        m = sums(nrm, aff.max() + 1)[aff]
        m /= np.linalg.norm(m, axis=1, keepdims=True)
        # directors are summed in steps of 2^-40, half a step each, and their sum is
        # at least half their number long
        assert np.minimum(np.abs(f - m).max(1), np.abs(f + m).max(1)).max() < 2.0 ** -40 + 1e-14
    sim.voronoi_update()
    c = np.asarray(sim.voronoi_get()[0], np.float64).reshape(-1, 3)
    cnt = np.bincount(aff, minlength=len(c))
    want = sums(x, len(c))[cnt > 0] / cnt[cnt > 0, None]
    # the mean to FP32, from positions summed in steps of 2^-32
    assert np.abs(c[cnt > 0] - want).max() <= 2.0 ** -24 * np.abs(want).max() + 2.0 ** -31
    sim.close()


@pytest.mark.parametrize("lost", [[0], [63], [5, 6, 777], list(range(128, 192))])
def test_partition_with_positions_that_are_not_numbers(lost):
    """Velocities that are not numbers carry positions with them; every other lipid
    finds its cell, and those keep theirs."""
    s = systems.planar_patch(40, 25, seed=5)
    v = np.zeros_like(s["lipid_x"])
    v[lost] = np.nan
    sim = orbc.Simulation(precision=orbc.FP64, skin=SKIN)
    sim.set_state(orbc.LIPID, s["lipid_x"], s["lipid_n"], s["lipid_id"], v=v)
    z = np.zeros((0, 3))
    sim.set_state(orbc.PROTEIN, z, z, np.zeros(0, np.uint32), type=np.zeros(0, np.int32))
    sim.voronoi_init(70, 2)
    before = sim.voronoi_get()[1]
    sim.integrate("verlet_langevin")
    x = sim.get_state(orbc.LIPID)["x"]
    assert np.array_equal(np.flatnonzero(np.isnan(x).any(1)), np.sort(lost))
    sim.voronoi_update()
    c, aff, _ = sim.voronoi_get()
    c = np.asarray(c, np.float32).reshape(-1, 3)
    ok = np.isfinite(x).all(1)
    with np.errstate(over="ignore"):
        assert np.array_equal(aff[ok], _nearest(c, x[ok]))
    assert np.array_equal(aff[~ok], before[~ok])
    sim.close()
