"""Device memory of the multi-level far field's work lists and partial sums."""
import ctypes
import gc

import numpy as np
import pytest

S = pytest.importorskip("spheresimulator_amd")

pytestmark = pytest.mark.gpu


def used():
    """Device memory in use, from the HIP runtime that libsphstk.so itself links."""
    S.load()
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return total.value - free.value


def test_coarse_set_holds_each_levels_own_partial_sums():
    """Coarse operator of 4096 spheres p=12: levels of 170 + 50 + 38 + 26 + 14 points
    per sphere behind the fine grid's 338, and source cells on the last two, 2.6e6
    targets in all.  A list wants 40000 items of 64 targets, so its partial sums
    (24 bytes each) take at most that or, with one slice, its own targets: 61 MB for
    each of the seven small lists and 33 MB for the fine grid.  With 72 bytes of
    records per point, intervals (48 bytes; about 5e6) and the matrices that is below
    1.1 GB; one slot count for all lists takes the 24 to 32 of the coarsest, 1.5 to 2 GB
    for the partial sums alone."""
    gc.collect()  # handles of earlier tests
    n = 4096
    c = S.configs.make_suspension(n, 12, 11, vf=0.1, min_gap=0.2)
    op = S.SphereSTKSHOperator(c["pos"], c["radius"], c["quat"], c["order"], 0.5, 0.0, 1.0, 1.0)
    x = np.random.default_rng(1).standard_normal(op.n_dof)
    op.apply_inner(x)  # code objects, the operator's own buffers
    before = used()
    y = op.apply_coarse(x)
    assert np.isfinite(y).all()
    assert used() - before < 1.1e9
