"""One lane per atom (launches over many tiles) and four lanes per atom with four workgroups
per tile (launches over at most 128 tiles) give the same bits: a system alone, and the same
system in a batch of copies whose class has more tiles, take the two routes.

Sizes at the edges: work items of a whole-box system (256 atoms each, 64 a part), two atoms,
lists whose groups do not fill a round of four lanes, mixtures, small boxes with a per-pair
image, sheared boxes, and FP64 forces of both routes against the oracle.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from pis_amd import Engine, plan, workloads as W
from tests.conftest import force_err
from tests.test_gpu_npt import sheared

pytestmark = pytest.mark.gpu

SYSTEMS = {
    "two_atoms": lambda: W.lj_box(2, 0.002, 1.0, seed=70),
    "whole_63": lambda: W.lj_box(63, 0.4, 1.0, seed=71),
    "whole_256": lambda: W.lj_box(256, 0.7, 1.0, seed=72),
    "whole_257": lambda: W.lj_box(257, 0.7, 1.0, seed=73),
    "whole_321_mixture": lambda: W.ka_mixture(321, 1.2, 1.0, seed=74),
    "raw_1500": lambda: W.lj_box(1500, 0.9, 1.0, seed=75),
    "tiled_4100_mixture": lambda: W.ka_mixture(4100, 1.2, 1.0, seed=76),
    "tiled_5000": lambda: W.lj_box(5000, 0.8, 1.2, seed=77),
    "sheared_2048": lambda: sheared(W.lj_liquid(8, 0.8442, 0.9, seed=78)),
    "sheared_500": lambda: sheared(W.lj_liquid(5, 0.8442, 0.9, seed=79)),
}


def work_items(spec, precision):
    p = plan(spec, precision)
    return -(-spec.n // 256) if p["mode"] == 2 else int(np.prod(p["ntile"]))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_one_and_four_lanes_give_the_same_bits(name, precision):
    spec = SYSTEMS[name]()
    tiles = work_items(spec, precision)
    copies = 128 // tiles + 1
    assert tiles <= 128 < tiles * copies
    print(f"{name} {precision}: N={spec.n}, {tiles} work items, {copies} copies", flush=True)
    got = []
    for specs in ([spec], [spec] * copies):
        with Engine(specs, precision) as eng:
            eng.load()
            pe = eng.compute_potential()
            f0 = eng.get_state(0)[2]
            th = eng.run_nve(spec.dt, 25)
            got.append((pe, f0, th, [eng.get_state(k) for k in range(len(specs))]))
    (pe1, f1, th1, st1), (pe4, f4, th4, st4) = got
    assert np.all(pe4 == pe1[0]) and np.array_equal(f1, f4)
    for k in range(copies):
        assert np.array_equal(th4[:, k], th1[:, 0])
        for a, b in zip(st4[k], st1[0]):
            assert np.array_equal(a, b)
    if precision == "fp64":
        o = po.OSystem.from_spec(spec)
        pe_ref = o.compute(po.MGR_BRUTE)
        assert abs(pe1[0] - pe_ref) <= 1e-12 * max(abs(pe_ref), 1.0)
        if np.abs(o.force).max() > 1e-6:
            assert force_err(f1, o.force) <= 1e-10
        else:  # a perfect lattice, or atoms out of reach: the forces vanish, no scale to relate to
            assert np.abs(f1 - o.force).max() <= 1e-10
