"""What a thermostat leaves to the next step is done in time for every reader."""

import ctypes

import numpy as np
import pytest

from halmd_amd import _lib, mdsim, workloads

pytestmark = pytest.mark.gpu

OPTIONS = {"verlet_nvt_hoover": dict(resonance_frequency=5.0), "verlet_nvt_andersen": dict(collision_rate=5.0)}


def _system(integrator, n):
    return workloads.lennard_jones(n, density=0.8442, temperature=1.2, jitter=0.02, seed=11, timestep=0.004,
                                   integrator=integrator, sort_interval=25, **OPTIONS[integrator])


# (not a multiple of a wave; several workgroups; more particles than the partial
# sums have threads)
@pytest.mark.parametrize("n", [1001, 4096, 70000])
@pytest.mark.parametrize("integrator", sorted(OPTIONS))
def test_reading_between_steps_leaves_the_trajectory(integrator, n):
    a, b = _system(integrator, n), _system(integrator, n)
    steps = 60
    a.sampler.run(steps)
    for k in range(steps):
        b.sampler.run(1)
        if k % 3 == 0:
            b.particle.data["velocity"]
        elif k % 7 == 1:
            b.particle.data["velocity"] = b.particle.data["velocity"]
        if integrator == "verlet_nvt_hoover" and k % 5 == 0:
            b.integrator.set_temperature(1.2)
            b.integrator.position
    if integrator == "verlet_nvt_andersen":
        # the same arithmetic in either kernel
        for name in ("position", "velocity", "image"):
            assert np.array_equal(a.particle.ordered(name), b.particle.ordered(name)), name
    else:
        # the sum of the rescaled velocities is taken from the one before: FP64
        # rounding in the scale, which can flip the last bit of a fixed-point
        # coordinate (L / 2^32 = 1e-8); with a curvature of 1e3 and dt = 0.004
        # that is 4e-8 in a velocity, which grows by a few e in 60 steps
        for name in ("position", "velocity"):
            assert np.max(np.abs(a.particle.ordered(name) - b.particle.ordered(name))) < 1e-6, name
        assert np.allclose(a.integrator.position, b.integrator.position, rtol=1e-6, atol=1e-12)
        assert np.allclose(a.integrator.velocity, b.integrator.velocity, rtol=1e-6, atol=1e-9)


def _assert_same(integrator, a, b):
    for name in ("position", "velocity", "image"):
        x, y = a.particle.ordered(name), b.particle.ordered(name)
        if integrator == "verlet_nvt_andersen":
            assert np.array_equal(x, y), name
        else:
            assert np.max(np.abs(x - y)) < 1e-6, name   # (as above)


@pytest.mark.parametrize("thermostat_first", [True, False])
@pytest.mark.parametrize("integrator", sorted(OPTIONS))
def test_second_integrator_on_the_particle(integrator, thermostat_first):
    # every half kick arrives, whichever integrator owes it
    runs = []
    for read in (False, True):
        w = _system(integrator, 1001)
        other = mdsim.integrators.verlet(box=w.box, particle=w.particle, timestep=0.002)
        order = [w.integrator, other] if thermostat_first else [other, w.integrator]
        for _ in range(8):
            for g in order:
                g.integrate()
            for g in order:
                g.finalize()
                if read:
                    w.particle.data["velocity"]
        runs.append(w)
    _assert_same(integrator, *runs)


def _replace_integrator(w):
    w.replaced = w.integrator   # (kept: its chain is still owed)
    w.integrator = mdsim.integrators.verlet(box=w.box, particle=w.particle, timestep=0.004)
    w.core.set_integrator(w.integrator)


def _write_positions(w):
    r = w.particle.data["position"]
    w.particle.data["position"] = np.roll(r, 1, axis=0)


def _write_mass(w):
    w.particle.data["mass"] = np.where(w.particle.data["id"] % 3 == 0, 2.0, 1.0)


def _add_force(w):
    soft = mdsim.potentials.pair.power_law(epsilon=0.1, sigma=1.0, index=6)
    w.second = mdsim.forces.pair_full(box=w.box, particle=w.particle, potential=soft)


@pytest.mark.parametrize("event", [_replace_integrator, _write_positions, _write_mass, _add_force])
@pytest.mark.parametrize("integrator", sorted(OPTIONS))
def test_changes_between_steps_come_after_what_is_owed(integrator, event):
    # the same change with the velocities read before it, which has everything done
    runs = []
    for read in (False, True):
        w = _system(integrator, 1001)
        w.sampler.run(7)
        if read:
            w.particle.data["velocity"]
        event(w)
        w.sampler.run(5)
        runs.append(w)
    _assert_same(integrator, *runs)


def test_profile_counts_andersen_collisions():
    # each step's collisions are launched by "integrate" (with the next step)
    # or by "finalize" (when the velocities are read first)
    w = _system("verlet_nvt_andersen", 1001)

    def launches(module):
        ms, n = ctypes.c_double(), ctypes.c_uint64()
        _lib.call("halmd_profile_collect", w.integrator.handle, module, ctypes.byref(ms), ctypes.byref(n))
        assert (ms.value > 0) == (n.value > 0)
        return n.value

    w.sampler.run(1)   # (the first step's half is made by the force kernel)
    for module in (b"integrate", b"finalize"):
        _lib.call("halmd_profile_enable", w.integrator.handle, module, 100)
    w.sampler.run(7)
    assert (launches(b"integrate"), launches(b"finalize")) == (7, 0)
    w.particle.data["velocity"]
    assert (launches(b"integrate"), launches(b"finalize")) == (0, 1)
    for _ in range(5):
        w.sampler.run(1)
        w.particle.data["velocity"]
    assert (launches(b"integrate"), launches(b"finalize")) == (5, 5)
