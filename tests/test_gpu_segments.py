"""Cell segments of any shape give the same lists and, where each particle's
force is summed in two streams (below 2^18 particles), the same trajectory."""

from types import SimpleNamespace

import numpy as np
import pytest
from forcecheck import force_errors

from halmd_amd import mdsim, workloads

pytestmark = pytest.mark.gpu

SHAPES = (None, (1, 1, 64), (2, 1, 128), (3, 2, 256))


def _system(kind, n, jitter):
    if kind == "ka":
        return workloads.kob_andersen(n, density=1.2, temperature=0.9, jitter=jitter, seed=5)
    return workloads.lennard_jones(n, density=0.8442, temperature=1.5, jitter=jitter, seed=5)


# 4 cells a side, some particles more than whole waves, two species; either side
# of the limit of the list build by three waves (104 * 1024)
@pytest.mark.parametrize("kind,n", [("lj", 1372), ("lj", 4001), ("ka", 8788), ("lj", 106495), ("lj", 106496)])
def test_shape_leaves_lists(oracle, kind, n):
    w = _system(kind, n, 0.15)
    for shape in SHAPES:
        if shape:
            w.neighbour.set_segments(*shape)
        w.neighbour.update()
        counts, entries = w.neighbour.lists()
        if shape is None:
            expect, lists, _ = oracle.staged_neighbour_list(
                w.particle.data["position_fixed"], w.particle.data["species"], w.neighbour.binning.ncell, w.length,
                w.potential.r_cut + w.skin, entries.shape[1])
        assert np.array_equal(counts, expect)
        valid = np.arange(entries.shape[1]) < counts[:, None]
        assert np.array_equal(entries[valid], lists[valid])


def _fullest(w):
    """Particles of the fullest segment."""
    nc, (S, R, _) = np.asarray(w.neighbour.binning.ncell, dtype=np.uint64), w.neighbour.segments
    c = (w.particle.data["position_fixed"].astype(np.uint64) * nc) >> np.uint64(32)
    return np.unique(np.stack([c[:, 0] // np.uint64(S), c[:, 1] // np.uint64(R), c[:, 2]]), axis=1,
                     return_counts=True)[1].max()


# (2^17: from here on segments of few particles are built by one lane each)
@pytest.mark.parametrize("n,shapes", [(4001, [(3, 1, 256), (2, 2, 256), (3, 2, 128)]),
                                      (32000, [(2, 2, 256), (5, 1, 256), (3, 2, 256)]),
                                      ((1 << 17) - 1, [(2, 1, 256), (3, 1, 256)]), (1 << 17, [(2, 1, 256), (3, 1, 256)])])
def test_lists_either_side_of_one_pass(oracle, n, shapes):
    # 128 particles: a pass of the list build by three waves; the fullest segment
    # of one build chooses the next one's kernel
    w = _system("lj", n, 0.15)
    w.neighbour.update()
    counts, entries = w.neighbour.lists()
    u, species = w.particle.data["position_fixed"], w.particle.data["species"]
    expect, lists, _ = oracle.staged_neighbour_list(u, species, w.neighbour.binning.ncell, w.length,
                                                    w.potential.r_cut + w.skin, entries.shape[1])
    valid = np.arange(entries.shape[1]) < expect[:, None]
    fullest = []
    for shape in shapes:
        w.neighbour.set_segments(*shape)
        fullest.append(_fullest(w))
        for _ in range(2):
            w.neighbour.update()
            counts, entries = w.neighbour.lists()
            assert np.array_equal(counts, expect)
            assert np.array_equal(entries[valid], lists[valid])
    assert min(fullest) <= 128 and (max(fullest) > 128 or n >= (1 << 17) - 1), fullest


@pytest.mark.parametrize("kind,n", [("lj", 1372), ("lj", 4001), ("ka", 8788), ("lj", 262143)])
def test_shape_leaves_trajectory(kind, n):
    runs = []
    for shape in SHAPES:
        w = _system(kind, n, 0.02)
        if shape:
            w.neighbour.set_segments(*shape)
        s = w.sampler.on_sample_thermodynamics(w.thermodynamics, 10)
        w.sampler.run(40)
        runs.append([w.particle.ordered(k) for k in ("position", "velocity", "image", "force")]
                    + [w.sampler.thermodynamics_records(s)])
    for r in runs[1:]:
        for a, b in zip(runs[0], r):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b)


def _boxed(n, edges, species, occupancy=0.4, seed=7):
    """n particles at random (a gradient along z) in a box of the given edge ratios, with lists."""
    edges = np.asarray(edges, dtype=np.float64)
    L = edges * (n / 0.8 / np.prod(edges)) ** (1.0 / 3)
    rng = np.random.default_rng(seed)
    u = rng.random((n, 3))
    u[:, 2] = u[:, 2] ** 1.15
    sp = (rng.random(n) < 0.3).astype(np.uint32) if species == 2 else np.zeros(n, np.uint32)
    kw = dict(epsilon=workloads.KA_EPSILON, sigma=workloads.KA_SIGMA) if species == 2 else dict(epsilon=1.0, sigma=1.0)
    pot = mdsim.potentials.pair.lennard_jones(**kw).truncate("shifted", cutoff=2.5)
    box = mdsim.box(length=L)
    p = mdsim.particle(dimension=3, particles=n, species=species)
    p.data["position"] = (u - 0.5) * L
    p.data["species"] = sp
    nb = mdsim.neighbour(particle=p, box=box, r_cut=pot.r_cut, skin=0.3, occupancy=occupancy, disable_sorting=True)
    return SimpleNamespace(length=L, box=box, particle=p, potential=pot, neighbour=nb, skin=0.3)


def _assert_lists(oracle, w):
    counts, entries = w.neighbour.lists()
    expect, lists, largest = oracle.staged_neighbour_list(
        w.particle.data["position_fixed"], w.particle.data["species"], w.neighbour.binning.ncell, w.length,
        w.potential.r_cut + w.skin, entries.shape[1])
    assert np.array_equal(counts, expect)
    valid = np.arange(entries.shape[1]) < counts[:, None]
    assert np.array_equal(entries[valid], lists[valid])
    return largest


# three different edges and odd numbers of cells (3 x 4 x 8 the fewest); lists
# larger than the capacity they start with (occupancy 1: the mean number); from
# one cell a segment to segments of two passes of the build by three waves, and
# (110,003) the build by one lane for each particle
@pytest.mark.parametrize("species", [1, 2])
@pytest.mark.parametrize("n,shapes", [(3001, [(1, 1, 64), (1, 2, 128)]), (20011, [(2, 2, 64), (4, 3, 256)]),
                                      (110003, [(2, 1, 256), (3, 2, 192)])])
def test_lists_in_a_box_of_three_edges(oracle, n, shapes, species):
    w = _boxed(n, (1.0, 1.31, 2.07), species, occupancy=1.0)
    nc = w.neighbour.binning.ncell
    assert len(set(int(x) for x in nc)) == 3, nc
    cap = w.neighbour.size
    fullest = []
    for shape in [None] + shapes:
        if shape:
            w.neighbour.set_segments(*shape)
        fullest.append(_fullest(w))
        for _ in range(2):   # (the second build goes by the first one's fullest segment)
            w.neighbour.update()
            assert _assert_lists(oracle, w) > cap
    assert w.neighbour.size > cap
    assert n < 20000 or (min(fullest) <= 128 < max(fullest)), fullest


@pytest.mark.parametrize("nspecies,n", [(1, 20011), (2, 3001), (2, 110003)])
def test_forces_in_a_box_of_three_edges(oracle, nspecies, n):
    # a displaced lattice: 4 particles a cubic cell, the cells of the box's edges
    edges = np.array([1.0, 1.31, 2.07])
    m = np.maximum(1, np.ceil(edges * (n / 4 / np.prod(edges)) ** (1.0 / 3))).astype(int)
    L = m * (4 / 0.8) ** (1.0 / 3)
    rng = np.random.default_rng(3)
    k = np.arange(4 * np.prod(m))
    base = np.array([[0.25, 0.25, 0.25], [0.75, 0.75, 0.25], [0.75, 0.25, 0.75], [0.25, 0.75, 0.75]])
    r = np.stack([(k >> 2) % m[0], ((k >> 2) // m[0]) % m[1], (k >> 2) // (m[0] * m[1])], axis=1) + base[k & 3]
    r = rng.permutation(r + rng.uniform(-0.08, 0.08, r.shape))[:n] * (L / m) - L / 2
    sp = (rng.random(n) < 0.3).astype(np.uint32) if nspecies == 2 else np.zeros(n, np.uint32)
    eps, sigma = (workloads.KA_EPSILON, workloads.KA_SIGMA) if nspecies == 2 else (1.0, 1.0)
    pot = mdsim.potentials.pair.lennard_jones(epsilon=eps, sigma=sigma).truncate("force_shifted", cutoff=2.5)
    box = mdsim.box(length=L)
    p = mdsim.particle(dimension=3, particles=n, species=nspecies)
    p.data["position"] = r
    p.data["species"] = sp
    nb = mdsim.neighbour(particle=p, box=box, r_cut=pot.r_cut, skin=0.3, disable_sorting=True)
    force = mdsim.forces.pair_trunc(box=box, particle=p, potential=pot, neighbour=nb)   # noqa: F841 (kept alive)
    p.data["force"]   # (the lists put the particles in cell order)
    ref = oracle.Potential(oracle.POT_LJ, "force_shifted", eps, sigma, 2.5)
    f, u = p.data["force"], p.data["potential_energy"]
    pos, species = p.data["position"], p.data["species"]
    fref, uref, _ = oracle.pair_force(pos, species, L, ref, skin=0.3)
    force_errors(f, fref, pos, species, L, ref, oracle, 1e-5)   # (asserts the bound of every particle)
    assert abs(u.sum() - uref.sum()) < 1e-6 * np.abs(uref).sum()


# cubic boxes of 4 cells a side and of more, one and two species
@pytest.mark.parametrize("species,n", [(1, 1200), (1, 20011), (2, 5003), (2, 110003)])
def test_windowed_build_gives_the_same_lists(oracle, monkeypatch, species, n):
    monkeypatch.setenv("HALMD_LIST_WINDOWS", "1")
    w = _boxed(n, (1.0, 1.0, 1.0), species, occupancy=1.0)
    assert min(w.neighbour.binning.ncell) >= 4
    cap = w.neighbour.size
    for shape in (None, (1, 1, 64), (2, 2, 256)):
        if shape:
            w.neighbour.set_segments(*shape)
        w.neighbour.update()
        assert _assert_lists(oracle, w) > cap
