"""Routes that a call takes by its size, each against the other route of the same call:

* a thermostatted or barostatted run with four lanes per atom (launches over at most 128 work
  items) and with one (the same system among enough copies);
* a host-driven run of a system large enough for one lane per atom against the fixed
  sequence of a batch, for each ensemble;
* a barostatted run whose grid is planned again on the way: every step has its record;
* states just below and just above what the pinned staging holds, and records beyond it.
"""
import tracemalloc

import numpy as np
import pytest

from oracle import pyoracle as po
from pis_amd import Atoms, Engine, LennardJones, LJGpuManager, plan, workloads as W
from tests.test_gpu_npt import sheared

pytestmark = pytest.mark.gpu

PINNED = 4 << 20  # bytes of the pinned staging
LANES_LIMIT = 128  # work items up to which a launch takes four lanes per atom


def work_items(spec, precision):
    p = plan(spec, precision)
    return -(-spec.n // 256) if p["mode"] == 2 else int(np.prod(p["ntile"]))


def run(specs, precision, ens, calls, system=0):
    with Engine(specs, precision) as eng:
        eng.load()
        eng.compute_potential()
        if ens == "nvt":
            eng.nvt_init(1.2, 0.9, 2.0)
        if ens == "npt":
            eng.npt_init(1.2, 0.9, 2.0, 1.0, 30.0)
        th, done = [], 0
        for k in calls:
            if ens == "nve":
                th.append(eng.run_nve(0.005, k))
            else:
                th.append({"nvt": eng.run_nvt, "npt": eng.run_npt}[ens](0.005, k, ramp=(done, sum(calls))))
            done += k
        box = eng.npt_box(system) if ens == "npt" else ()
        return np.concatenate(th)[:, system], eng.get_state(system), box, eng.stats()["rebuilds"] // len(specs)


def assert_same(a, b):
    assert np.array_equal(a[0], b[0])
    for x, y in zip(a[1] + tuple(a[2]), b[1] + tuple(b[2])):
        assert np.array_equal(x, y)
    assert a[3] == b[3]


LANE_SYSTEMS = {
    "whole_321_mixture": lambda: W.ka_mixture(321, 1.2, 1.0, seed=84),
    "raw_1500": lambda: W.lj_box(1500, 0.9, 1.0, seed=85),
    "tiled_4100_mixture": lambda: W.ka_mixture(4100, 1.2, 1.0, seed=86),
    "tiled_5000": lambda: W.lj_box(5000, 0.8, 1.2, seed=87),
    "sheared_2048": lambda: sheared(W.lj_liquid(8, 0.8442, 0.9, seed=88)),
}


@pytest.mark.parametrize("ens", ["nvt", "npt"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", sorted(LANE_SYSTEMS))
def test_one_and_four_lanes_agree_under_a_thermostat_and_a_barostat(name, precision, ens):
    spec = LANE_SYSTEMS[name]()
    tiles = work_items(spec, precision)
    copies = LANES_LIMIT // tiles + 1
    assert tiles <= LANES_LIMIT < tiles * copies
    print(f"{name} {precision} {ens}: N={spec.n}, {tiles} work items, {copies} copies", flush=True)
    assert_same(run([spec], precision, ens, [12, 13]), run([spec] * copies, precision, ens, [12, 13], copies - 1))


@pytest.mark.parametrize("ens", ["nve", "nvt", "npt"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_driven_run_of_a_large_system_equals_the_fixed_sequence(precision, ens):
    spec = W.lj_liquid(20, 0.8442, 1.2, seed=89, skin=0.15)
    tiles = work_items(spec, precision)
    assert tiles > LANES_LIMIT  # one lane per atom, alone or in a batch
    a = run([spec], precision, ens, [3, 40])
    print(f"{precision} {ens}: N={spec.n}, {tiles} work items, {a[3]} rebuilds", flush=True)
    assert a[3] >= 3
    assert_same(a, run([spec, spec], precision, ens, [3, 40]))


def test_a_run_that_is_planned_again_on_the_way_has_every_record():
    """The box shrinks below its cell grid within a call (the oracle crosses it at step 57): the
    steps before and after the new plan are all there and track the oracle, and one call
    gives the records of shorter ones."""
    def new():
        return W.lj_liquid(8, 0.8442, 0.9, seed=66, rcut=2.5, skin=0.3, dt=0.004)

    def go(calls):
        spec = new()
        with Engine(spec, "fp64") as eng:
            eng.load()
            eng.compute_potential()
            eng.npt_init(0.9, 0.9, 0.5, 12.0, 8.0, 3)
            th, done = [], 0
            for k in calls:
                th.append(eng.run_npt(spec.dt, k, ramp=(done, sum(calls)))[:, 0])
                done += k
            return np.concatenate(th), eng.compute_potential()[0], eng.get_state(0), eng.stats()

    th, pe, st, stats = go([120])
    assert th.shape == (120, 7) and np.all(np.isfinite(th)) and np.all(th[:, 3] > 0)
    spec = new()
    ref, _ = po.OSystem.from_spec(spec).run_npt(spec.dt, 120, 0.9, 0.9, 0.5, 12.0, 8.0, 3, kb=spec.kb)
    assert np.abs(th[:, :3] - ref[:, :3]).max() <= 1e-8 * np.abs(ref[:, 0]).max()
    th2, pe2, st2, _ = go([20, 45, 1, 54])
    # the grid is planned at the same step either way; chunks of 64 steps only end elsewhere
    assert np.abs(th - th2).max() <= 1e-8 * np.abs(th).max()
    assert abs(pe - th[-1, 0]) <= 1e-12 * abs(pe)  # the list that the run left behind is whole
    assert stats["steps"] == 120
    assert stats["force_launches"] == 120 + 2  # a force launch a step, and the two force calls


def state_of(n, seed):
    rng = np.random.default_rng(seed)
    spec = W.lj_box(n, 0.8442, 1.0, seed=seed)
    return spec, rng.normal(size=(n, 3)), rng.normal(size=(n, 3))


# upload: 73 bytes per atom in one piece; download: 24 per atom for each of the arrays asked for
@pytest.mark.parametrize("n", [PINNED // 73, PINNED // 73 + 1, PINNED // 72, PINNED // 72 + 1,
                               PINNED // 24, PINNED // 24 + 1])
def test_states_around_the_pinned_staging_come_back_whole(n):
    spec, vel, frc = state_of(n, 91)
    print(f"N={n}", flush=True)
    with Engine(spec, "mixed") as eng:
        for k in range(2):  # the second with the staging grown, and with other values
            eng.set_state(0, spec.positions, vel + k, frc - k)
            p, v, f = eng.get_state(0)
            assert np.array_equal(p, spec.positions) and np.array_equal(v, vel + k) and np.array_equal(f, frc - k)
            assert np.array_equal(eng.get_forces(0), frc - k)
            assert np.array_equal(eng.get_positions(0), spec.positions)
        eng.set_state(0, spec.positions)  # no velocities, no forces: zero
        p, v, f = eng.get_state(0)
        assert np.array_equal(p, spec.positions) and not v.any() and not f.any()


# 12 bytes per atom come back
@pytest.mark.parametrize("n", [2, 4000, PINNED // 12, PINNED // 12 + 1])
def test_list_digests_around_the_pinned_staging_match_the_list(n):
    spec = W.lj_box(n, 0.3 if n > 2 else 0.002, 1.0, seed=93)
    with Engine(spec, "mixed") as eng:
        eng.load()
        counts, hashes = eng.list_digest()
        offsets, idx = eng.neighbor_list()
        again = eng.list_digest()
    assert np.array_equal(counts, np.diff(offsets))
    with np.errstate(over="ignore"):  # splitmix64's output function, summed over each row
        x = idx.astype(np.uint64) + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        x ^= x >> np.uint64(31)
        total = np.concatenate([np.zeros(1, dtype=np.uint64), np.cumsum(x, dtype=np.uint64)])
        assert np.array_equal(hashes, total[offsets[1:]] - total[offsets[:-1]])
    assert np.array_equal(again[0], counts) and np.array_equal(again[1], hashes)


@pytest.mark.parametrize("n", [4000, PINNED // 72 + 1, 262144])
def test_per_call_steps_and_forces_make_no_arrays(n):
    """The drop-in calls bring the state back through arrays that the manager keeps: made anew
    for each call they are fresh pages, or not, by what the process's heap happens to keep."""
    spec = W.lj_box(n, 0.8442, 1.0, seed=92)
    mgr = LJGpuManager(skin=spec.skin, kb=spec.kb, precision="mixed")
    for ti, tj, eps, sig, rc in spec.pairs:
        mgr.insert((ti, tj), LennardJones(eps, sig, rc, True))
    atoms = Atoms(spec.type_ids, spec.masses, spec.positions, spec.velocities, spec.box)
    mgr.compute_potential(atoms)
    mgr.verlet_step_nve(atoms, spec.dt)
    tracemalloc.start()
    try:
        for call in (lambda: mgr.verlet_step_nve(atoms, spec.dt), lambda: mgr.compute_potential(atoms)):
            tracemalloc.reset_peak()
            base = tracemalloc.get_traced_memory()[0]
            call()
            peak = tracemalloc.get_traced_memory()[1] - base
            print(f"N={n}: {peak} bytes at most", flush=True)
            assert peak < 24 * n  # less than one array of the state (the engine's key takes 4 n)
    finally:
        tracemalloc.stop()
    # and the arrays are the atoms' own: another set of atoms does not see them
    other = Atoms(spec.type_ids, spec.masses, spec.positions, spec.velocities, spec.box)
    kept = atoms.positions.copy(), atoms.velocities.copy(), atoms.forces.copy()
    mgr.compute_potential(other)
    mgr.verlet_step_nve(other, spec.dt)
    for a, b in zip(kept, (atoms.positions, atoms.velocities, atoms.forces)):
        assert np.array_equal(a, b)


def test_records_beyond_the_pinned_staging_equal_those_within_it():
    specs = [W.lj_box(64, 0.3, 1.0, seed=100 + k) for k in range(300)]
    steps = PINNED // (56 * len(specs)) + 20
    got = []
    for calls in ([steps], [steps // 3, steps // 3, steps - 2 * (steps // 3)]):
        assert (max(calls) * 56 * len(specs) > PINNED) == (len(calls) == 1)
        with Engine(specs, "mixed") as eng:
            eng.load()
            eng.compute_potential()
            got.append(np.concatenate([eng.run_nve(0.002, k) for k in calls]))
    print(f"{steps} records of {len(specs)} systems", flush=True)
    assert np.array_equal(*got)
