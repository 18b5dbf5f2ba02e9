"""Levels of a multi-level far field that are some spheres' own grids: orders at
and around those of the levels, mixed in one handle, down to handles where every
level is everyone's own grid."""
import numpy as np
import pytest

S = pytest.importorskip("spheresimulator_amd")

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def spread(orders, n, seed, gap, c=(0.5, 0.0, 1.0, 1.0), **kw):
    """n spheres along a line, next ones `gap` apart, so that pairs lie on every level."""
    r = np.random.default_rng(seed)
    rad = 0.8 + 0.4 * r.random(n)
    z = np.cumsum(2 * rad + gap)
    pos = np.stack([0.4 * np.sin(z), 0.4 * np.cos(z), z], 1)
    return S.SphereSTKSHOperator(pos, rad, S.configs.Stream(seed).quaternions(n),
                                 np.resize(np.array(orders, dtype=np.int32), n), *c, **kw), r


@pytest.mark.parametrize("cells", [True, False])
@pytest.mark.parametrize("orders", [(1, 2, 3), (2, 16), (4, 5, 6), (5, 10, 11), (6, 8, 10, 12, 16), (3, 20)])
def test_rough_densities_on_mixed_orders(orders, cells):
    """Rough densities (no projection): a sphere's own grid carries all of it.  Bounds
    of the operators on random packings (outer 2e-9, inner 5e-5, coarse 5e-2); on own
    grids alone the FP32 operator is FP32 sums: 2e-6."""
    op, r = spread(orders, 60, len(orders), 1.0, cells=cells)
    x = r.standard_normal(op.n_dof)
    y = op.apply(x)
    assert rel(op.apply_outer(x), y) < 2e-9
    assert rel(op.apply_inner(x), y) < (2e-6 if max(orders) <= 3 else 5e-5)
    assert rel(op.apply_coarse(x), y) < 5e-2


def test_small_orders_alone_are_exact_in_the_fp64_levels():
    """Orders up to 5: every level of the FP64 set is the own grid of all spheres, for
    all four coefficients."""
    op, r = spread((3, 4, 5), 80, 9, 0.5, (0.3, 0.7, 1.1, 0.9))
    x = r.standard_normal(op.n_dof)
    assert rel(op.apply_outer(x), op.apply(x)) < 1e-13


def test_batch_with_finished_suspensions():
    """Mixed solve of suspensions of orders 4, 8 and 12 that converge after different
    numbers of steps, against each alone: the refinement's tolerance of 1e-8 on both."""
    parts = [S.configs.make_suspension(n, p, 20 + p, vf=0.05, min_gap=0.2) for n, p in ((30, 4), (70, 8), (40, 12))]
    c = {k: np.concatenate([q[k] for q in parts]) for k in ("pos", "radius", "quat", "order", "force")}
    both = S.SphereSTKMobMat(c["pos"], c["radius"], c["quat"], c["order"], counts=[30, 70, 40],
                             precision=S.PREC_MIXED)
    v, info = both.solveMob(c["force"])
    at = 0
    for q in parts:
        one = S.SphereSTKMobMat(q["pos"], q["radius"], q["quat"], q["order"], precision=S.PREC_MIXED)
        w, _ = one.solveMob(q["force"])
        assert rel(v[at:at + len(w)], w) < 1e-7
        at += len(w)
