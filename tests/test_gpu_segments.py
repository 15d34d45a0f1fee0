"""Cell segments of any shape give the same lists and, where each particle's
force is summed in two streams (below 2^18 particles), the same trajectory."""

import numpy as np
import pytest

from halmd_amd import workloads

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
