"""A single system's steps are driven by the host (list rebuilds launched when a step reports
one due); a batch runs the fixed sequence with the rebuild kernels in every step.  Both give
the same bits, records and rebuild counts.

The cases are the edges of the drive: runs shorter than the steps queued ahead, a skin so
thin that nearly every step rebuilds, no skin at all, a rebuild due in a call's first step,
runs continued over several calls, NVT (whose position update finds the due rebuild) and NPT
(whose second half runs behind the step)."""
import numpy as np
import pytest

from pis_amd import Engine, PisError, workloads as W

pytestmark = pytest.mark.gpu


def spec_with(skin, n=1372, temp=1.5):
    s = W.lj_box(n, 0.85, temp, seed=90, skin=skin)
    s.positions = s.positions + np.random.default_rng(5).uniform(-0.03, 0.03, s.positions.shape)
    s.positions = W.wrap_positions(s.positions, s.box.lengths)
    return s


def run(specs, precision, calls, ens):
    with Engine(specs, precision) as eng:
        eng.load()
        eng.compute_potential()
        if ens == "nvt":
            eng.nvt_init(1.5, 1.0, 2.0)
        if ens == "npt":
            eng.npt_init(1.5, 1.0, 2.0, 1.0, 30.0)
        th = []
        done = 0
        for k in calls:
            step = {"nve": eng.run_nve, "nvt": eng.run_nvt, "npt": eng.run_npt}[ens]
            th.append(step(0.005, k) if ens == "nve" else step(0.005, k, ramp=(done, sum(calls))))
            done += k
        return np.concatenate(th)[:, 0], eng.get_state(0), eng.stats()["rebuilds"] // len(specs)


@pytest.mark.parametrize("ens", ["nve", "nvt", "npt"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("skin,calls", [(0.3, [1]), (0.3, [2, 1]), (0.3, [3, 4, 5]), (0.3, [60]), (0.02, [1, 2, 20]),
                                        (0.0, [7]), (0.15, [31, 1, 1, 17])],
                         ids=lambda v: str(v))
def test_driven_run_equals_the_fixed_sequence(skin, calls, precision, ens):
    spec = spec_with(skin)
    th1, st1, r1 = run([spec], precision, calls, ens)
    th2, st2, r2 = run([spec, spec], precision, calls, ens)
    print(f"skin {skin} calls {calls} {precision} {ens}: {r1} rebuilds", flush=True)
    assert np.array_equal(th1, th2)
    for a, b in zip(st1, st2):
        assert np.array_equal(a, b)
    assert r1 == r2
    if skin <= 0.02:
        assert r1 >= sum(calls)  # the state's own list and one nearly every step


def test_driven_run_reports_a_blown_up_system():
    """Non-finite positions end the run with the error the fixed sequence gives, not a wait."""
    spec = spec_with(0.3)
    bad = spec.velocities.copy()
    bad[3] = np.nan
    with Engine(spec, "fp64") as eng:
        eng.load()
        eng.compute_potential()
        eng.set_state(0, spec.positions, bad, np.zeros_like(bad))
        with pytest.raises(PisError) as e:
            eng.run_nve(0.005, 20)
        assert e.value.name == "PIS_ERR_NAN_ENERGY"
