"""A host-driven run whose thread shares its CPU with others: steps queued with their rebuild
launches while the thread is late give the bits of an undisturbed run, for each ensemble, in
one call and in short ones, and the device does not wait for the thread at every rebuild."""
import os
import subprocess
import sys
import threading
import time

import numpy as np
import pytest

from pis_amd import Engine, workloads as W

pytestmark = pytest.mark.gpu

HOG = ("import os, sys, time\nos.sched_setaffinity(0, {int(sys.argv[1])})\nprint('on', flush=True)\n"
       "t = time.time()\nwhile time.time() - t < 30: pass\n")


class BusyCpu:
    """Pins the calling thread to one CPU that `others` busy processes share."""

    def __init__(self, others=3):
        self.others = others

    def __enter__(self):
        self.cpus = os.sched_getaffinity(0)
        cpu = max(self.cpus)
        self.procs = [subprocess.Popen([sys.executable, "-c", HOG, str(cpu)], stdout=subprocess.PIPE)
                      for _ in range(self.others)]
        for p in self.procs:
            p.stdout.readline()
        os.sched_setaffinity(0, {cpu})
        return self

    def __exit__(self, *exc):
        os.sched_setaffinity(0, self.cpus)
        for p in self.procs:
            p.kill()
        for p in self.procs:
            p.wait()
            p.stdout.close()


def run(spec, precision, ens, calls, busy, timed=False):
    with Engine(spec, precision) as eng:
        eng.load()
        eng.compute_potential()
        if ens == "nvt":
            eng.nvt_init(1.2, 1.0, 2.0)
        if ens == "npt":
            eng.npt_init(1.2, 1.0, 2.0, 1.0, 30.0)
        eng.set_kernel_timing(timed)  # steps of the fixed sequence

        def steps():
            th, done = [], 0
            for k in calls:
                if ens == "nve":
                    th.append(eng.run_nve(0.005, k))
                else:
                    th.append({"nvt": eng.run_nvt, "npt": eng.run_npt}[ens](0.005, k, ramp=(done, sum(calls))))
                done += k
            return np.concatenate(th)

        t0 = time.perf_counter()
        if busy:
            with BusyCpu():
                t0 = time.perf_counter()
                th = steps()
                sec = time.perf_counter() - t0
        else:
            th = steps()
            sec = time.perf_counter() - t0
        return sec, (th, *eng.get_state(0), eng.stats()["rebuilds"])


@pytest.mark.parametrize("ens,calls", [("nve", [1500]), ("nve", [40] * 20), ("nvt", [1200]), ("npt", [700])])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_late_thread_changes_no_bit(ens, calls, precision):
    spec = W.lj_liquid(10, 0.8442, 1.2, seed=95, skin=0.15)
    quiet, a = run(spec, precision, ens, calls, False)
    busy, b = run(spec, precision, ens, calls, True)
    print(f"{precision} {ens}: {a[-1]} rebuilds, {quiet * 1e3:.1f} ms, busy {busy * 1e3:.1f} ms", flush=True)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


def test_more_runs_than_cpus_change_no_bit():
    """One engine per thread, more of them than CPUs, several calls each."""
    spec = W.lj_liquid(8, 0.8442, 1.2, seed=97, skin=0.15)
    calls = [150, 40, 150]
    count = min(len(os.sched_getaffinity(0)) + 4, 24)
    _, alone = run(spec, "mixed", "nve", calls, False)
    out = [None] * count
    start = threading.Barrier(count)

    def work(k):
        start.wait()
        out[k] = run(spec, "mixed", "nve", calls, False)[1]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(count)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print(f"{count} runs", flush=True)
    for got in out:
        for x, y in zip(alone, got):
            assert np.array_equal(x, y)


def test_a_late_thread_does_not_stop_the_device():
    """262,144 atoms, a rebuild in every eighth step or so: the fixed sequence runs without the
    thread, and a driven run on the same busy CPU takes less than twice its time (1/4 of the
    CPU, and a wait for the thread at every rebuild, would take about four times)."""
    spec = W.lj_liquid(40, 0.8442, 1.0, seed=96)
    calls = [400] * 3
    driven = fixed = np.inf
    for _ in range(3):
        sec, a = run(spec, "mixed", "nve", calls, True)
        driven = min(driven, sec)
        sec, b = run(spec, "mixed", "nve", calls, True, timed=True)
        fixed = min(fixed, sec)
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
    print(f"driven {driven * 1e3:.1f} ms, fixed sequence {fixed * 1e3:.1f} ms, {a[-1]} rebuilds", flush=True)
    assert driven < 2.0 * fixed
