"""The largest systems that the allocation-free entry point's fixed scratch holds: one more
64-atom row of arrays is refused, and at the limit it gives the allocating route's bits."""
import numpy as np
import pytest

from pis_amd import workloads as W
from tests.test_zz_no_alloc import allocating, noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,density", [(121216, 0.8442), (200640, 0.1), (105920, 1.1)])
def test_the_largest_system_of_the_scratch(n, density):
    spec = W.lj_box(n, density, 1.0, seed=3)
    print(f"N={n} density {density}", flush=True)
    f_ref, pe_ref = allocating(spec, "mixed")
    st, f, pe = noalloc(spec, "mixed")
    assert st == 0
    assert np.array_equal(f, f_ref) and pe == pe_ref
    st, _, _ = noalloc(W.lj_box(n + 64, density, 1.0, seed=3), "mixed")
    assert st == 10  # PIS_ERR_CAPACITY
