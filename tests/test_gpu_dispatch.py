"""The sizes at which a kernel or its launch shape changes, against plain numpy or
against the path the other sizes take: sorts of one and several scan tiles, block
halos with two and four threads a row, the minimiser's fused step, cell sums of one
to four rounds, the warm partition of far-apart and scattered lipids, the cleanup of
cells with more members than a wave has lanes, and the thermostat's friction and the
volume push summed by the kernels that use them or by one of their own."""
import numpy as np
import pytest

import openrbc_amd as orbc
from openrbc_amd import systems

pytestmark = pytest.mark.gpu


def _no_proteins(sim):
    z = np.zeros((0, 3))
    sim.set_state(orbc.PROTEIN, z, z, np.zeros(0, np.uint32), type=np.zeros(0, np.int32))


def _lipids(x, n=None, seed=1, v=True, **kw):
    rng = np.random.default_rng(seed)
    if n is None:
        n = rng.normal(size=x.shape)
        n /= np.linalg.norm(n, axis=1, keepdims=True)
    sim = orbc.Simulation(seed=seed, **kw)
    sim.set_state(orbc.LIPID, x, n, np.arange(len(x), dtype=np.uint32), v=rng.normal(0, 0.3, x.shape) if v else None)
    _no_proteins(sim)
    return sim


def _patch(nx, ny, **kw):
    s = systems.planar_patch(nx, ny, seed=5)
    return _lipids(s["lipid_x"], s["lipid_n"], **kw)


# 2048 keys a sort tile, 4096 counters a scan tile: 16 tiles of 256 bins fill one
@pytest.mark.parametrize("n", [1, 2047, 2049, 16 * 2048, 16 * 2048 + 1, 700001])
@pytest.mark.parametrize("bits", [3, 8, 13, 32])
def test_sort_tiles(n, bits):
    rng = np.random.default_rng(n + bits)
    k = rng.integers(0, 1 << bits, n, dtype=np.uint32) if bits < 32 else rng.integers(0, 2**32, n, dtype=np.uint32)
    v = np.arange(n, dtype=np.uint32)
    with orbc.Simulation() as sim:
        ks, vs = sim.sort_pairs(k, v, bits)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(ks, k[order]) and np.array_equal(vs, v[order])


# 512 blocks of 256: four threads a row up to there, two beyond
@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
@pytest.mark.parametrize("nx,ny", [(5, 50), (256, 512), (257, 512)])
def test_halo_rows_shared(nx, ny, precision):
    out = []
    for halo in (2, 0):
        sim = _patch(nx, ny, precision=precision, block_halo=halo, skin=0.4)
        sim.run(4)
        out.append(sim.get_state(orbc.LIPID))
        if halo:
            assert sim.observables()["halo_blocks"] == -(-nx * ny // 256)
        sim.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k


@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
@pytest.mark.parametrize("nx,ny", [(15, 17), (16, 16), (1, 257)])
def test_minimize_batches(nx, ny, precision):
    """Any split of the steps into calls gives the same bits, through rebuilds and
    walls; velocities turn at a wall."""
    states = []
    for calls in ((23,), (1,) * 23, (2, 9, 12)):
        s = systems.planar_patch(nx, ny, a=0.95, seed=5)
        sim = _lipids(s["lipid_x"], s["lipid_n"], precision=precision, skin=0.1, box_lo=[0.0, -50.0, -50.0],
                      box_hi=[60.0, 60.0, 50.0])
        for c in calls:
            sim.minimize(c)
        states.append((sim.get_state(orbc.LIPID), sim.observables()["rebuilds"]))
        f, t = sim.get_forces(orbc.LIPID)[:2]
        assert not f.any() and not t.any()
        sim.close()
    for st, rb in states[1:]:
        assert rb == states[0][1]
        for k in st:
            assert np.array_equal(st[k], states[0][0][k]), k


@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
def test_minimize_step_from_forces(precision):
    """One step is the capped descent along the public forces (src/openrbc.cpp:114-131).
    The forces are read as the step has them (FP32 numbers in mixed precision); ten
    roundings of numbers up to 20 lie between, so 1e-13 is ten times what they add."""
    s = systems.planar_patch(20, 20, a=0.95, seed=5)
    x, n = s["lipid_x"], s["lipid_n"]
    sim = _lipids(x, n, precision=precision)
    sim.compute_pairwise(zero_first=True)
    sim.compute_bonded()
    f, t = sim.get_forces(orbc.LIPID)[:2]
    q = np.cross(n, t)
    if precision == orbc.MIXED:
        q = q.astype(np.float32).astype(np.float64)
    d = np.cross(q, n)
    a, b = np.linalg.norm(f, axis=1, keepdims=True), np.linalg.norm(d, axis=1, keepdims=True)
    h = np.where((a > 5e-2) | (b > 5e-2), np.minimum(5e-2 / a, 5e-2 / b), sim.cfg.dt)
    sim.minimize(1)
    got = sim.get_state(orbc.LIPID)
    m = n + d * h
    assert np.abs(got["x"] - (x + f * h)).max() < 1e-13
    # an FP32 rounding of n x t the other way moves a director by 6e-8 of its step
    tol = 1e-13 if precision == orbc.FP64 else 1e-8
    assert np.abs(got["n"] - m / np.linalg.norm(m, axis=1, keepdims=True)).max() < tol
    sim.close()


def _nearest(c, x):
    """Nearest centroid in FP32, lowest index on equal distance, as the partition has it."""
    p, out = x.astype(np.float32), np.empty(len(x), np.int64)
    for i in range(0, len(x), 512):
        d = p[i:i + 512, None, :] - c[None]
        d = d * d
        out[i:i + 512] = np.argmin((d[..., 0] + d[..., 1]) + d[..., 2], axis=1)
    return out


@pytest.mark.parametrize("case", ["pair of clusters", "scattered", "line", "lone cell"])
def test_partition_of_scattered_lipids(case):
    rng = np.random.default_rng(3)
    if case == "pair of clusters":            # waves that lie in two places
        x = np.concatenate([rng.uniform(-9, 9, (700, 3)), rng.uniform(-9, 9, (333, 3)) + [90, 40, -70]])
        cells = 60
    elif case == "scattered":                 # boxes of more cells than are staged
        x, cells = rng.uniform(-110, 110, (1500, 3)), 300
    elif case == "line":
        x, cells = np.stack([np.linspace(-200, 200, 999), np.zeros(999), np.zeros(999)], 1), 71
    else:
        x, cells = rng.uniform(-4, 4, (130, 3)), 1
    sim = _lipids(x, v=False, skin=0.4)
    sim.voronoi_init(cells, 2)
    for _ in range(2):
        sim.voronoi_update()
        c, aff, _ = sim.voronoi_get()
        assert np.array_equal(aff, _nearest(np.asarray(c, np.float32).reshape(-1, 3), sim.get_state(orbc.LIPID)["x"]))
    sim.close()


# blocks of 256 lipids: one round below 1800, two below 3600, then four
@pytest.mark.parametrize("blocks", [1, 57, 1799, 1801, 3601])
def test_cell_sum_rounds(blocks):
    n = blocks * 256 - 3
    nx = int(np.ceil(np.sqrt(n)))
    s = systems.planar_patch(nx, -(-n // nx), seed=5)
    x = s["lipid_x"][:n]
    sim = _lipids(x, s["lipid_n"][:n], v=False, skin=0.4)
    sim.voronoi_init(0, 0)
    old, aff, _ = sim.voronoi_get()
    sim.voronoi_update()
    c = np.asarray(sim.voronoi_get()[0], np.float64).reshape(-1, 3)
    cnt = np.bincount(aff, minlength=len(c))
    want = np.stack([np.bincount(aff, x[:, d], len(c)) for d in range(3)], 1)
    some = cnt > 0
    want = want[some] / cnt[some, None]
    # the mean to FP32, from positions summed in steps of 2^-32
    assert np.abs(c[some] - want).max() <= 2.0 ** -24 * np.abs(want).max() + 2.0 ** -31
    sim.close()


@pytest.mark.parametrize("cells", [1, 3, 40])
def test_cleanup_of_large_cells(cells):
    """Cells with up to 500 members: those not below tol^2 times the member distance
    of rank size / 2 go."""
    rng = np.random.default_rng(4)
    x = rng.normal(0, 12, (501, 3))
    sim = _lipids(x, v=False, skin=0.4)
    sim.voronoi_init(cells, 4)
    c, aff, _ = sim.voronoi_get()
    d2 = ((x - np.asarray(c, np.float64).reshape(-1, 3)[aff]) ** 2).sum(1)
    keep = np.ones(len(x), bool)
    for k in range(cells):
        m = np.flatnonzero(aff == k)
        if len(m):
            keep[m] = d2[m] < np.sort(d2[m])[len(m) // 2] * 1.7 ** 2
    assert 0 < (~keep).sum()
    assert sim.delete_stray_lipids(1.7) == (~keep).sum()
    assert np.array_equal(sim.get_state(orbc.LIPID)["x"], x[keep])
    sim.close()


# 1024 partial sums: up to there the halves sum them themselves
@pytest.mark.parametrize("precision", [orbc.MIXED, orbc.FP64])
@pytest.mark.parametrize("nx,ny", [(4, 63), (16, 16), (512, 512), (513, 512)])
def test_friction_in_the_halves(nx, ny, precision, monkeypatch):
    out = []
    for per_step in ("0", "1"):
        monkeypatch.setenv("ORBC_NH_PER_STEP", per_step)
        sim = _patch(nx, ny, precision=precision, skin=0.3, thermostat=orbc.RUN_NOSE_HOOVER)
        for k in (1, 9, 4):
            sim.run(k)
        out.append((sim.get_state(orbc.LIPID), sim.observables()))
        sim.close()
    assert out[0][1]["zeta"] == out[1][1]["zeta"] != 0
    for k in out[0][0]:
        assert np.array_equal(out[0][0][k], out[1][0][k]), k


# 64 partial sums of the volume, 256 cells each: up to there the step adds them up
@pytest.mark.parametrize("cells", [300, 64 * 256, 64 * 256 + 1])
def test_volume_push_in_the_step(cells):
    s = systems.init_rbc(*systems.geodesic(8 if cells > 300 else 2), rho=1.05, seed=7)
    states = []
    for staged in (False, True):
        sim = orbc.Simulation(precision=orbc.FP64, seed=3, skin=0.4, volume_target=0.0 if staged else -1.0,
                              volume_strength=0.5, freq_cleanup=0)
        sim.set_state(orbc.LIPID, s["lipid_x"], s["lipid_n"], s["lipid_id"])
        sim.set_state(orbc.PROTEIN, s["protein_x"], s["protein_n"], s["protein_id"], type=s["protein_type"])
        sim.set_bonds(s["bond_type"], s["bond_i"], s["bond_j"])
        sim.voronoi_init(cells, 1)
        if staged:
            target = sim.constrain_volume(1.0, 0.0)
            for step in range(3):
                if step % 2 == 0:
                    sim.voronoi_update()
                sim.compute_pairwise(zero_first=True)
                sim.compute_bonded()
                sim.constrain_volume(target, 0.5)
                sim.integrate("verlet_langevin")
        else:
            sim.run(3)
        states.append([sim.get_state(k) for k in (orbc.LIPID, orbc.PROTEIN)])
        sim.close()
    # the forces of the unrelaxed start reach some 1e3 and their terms are ordered differently
    # in the two paths: 1e-13 of that, over three steps of 0.01
    for a, b in zip(*states):
        for k in ("x", "v"):
            assert np.abs(a[k] - b[k]).max() < 1e-10, k
