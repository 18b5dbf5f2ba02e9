"""Which pairs the coarse operator sums on which grid: a matter of the two
spheres' orders and radii alone."""
import numpy as np
import pytest

S = pytest.importorskip("spheresimulator_amd")

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def density(op, seed):
    x = np.random.default_rng(seed).standard_normal(op.n_dof)
    op.projectNullSpace(x)
    return x


def test_coarse_operator_of_a_suspension_does_not_depend_on_the_batch():
    """64 spheres of order 8 alone, and in one handle with 4 spheres of order 12:
    the same pairs on the same grids, so the same sums up to the FP32 pair sums'
    rounding (1e-7 each) in another order of adding."""
    a = S.configs.make_suspension(64, 8, 3, vf=0.1, min_gap=0.2)
    b = S.configs.make_suspension(4, 12, 4, vf=0.05, min_gap=0.2)
    one = S.SphereSTKSHOperator(a["pos"], a["radius"], a["quat"], a["order"], 0.5, 0.0, 1.0, 1.0)
    two = S.SphereSTKSHOperator(*(np.concatenate([a[k], b[k]]) for k in ("pos", "radius", "quat", "order")),
                                0.5, 0.0, 1.0, 1.0, counts=[64, 4])
    x = density(two, 5)
    y1, y2 = one.apply_coarse(x[:one.n_dof]), two.apply_coarse(x)[:one.n_dof]
    assert rel(y1, one.apply(x[:one.n_dof])) > 1e-5  # (levels are in use)
    assert rel(y2, y1) < 1e-6


@pytest.mark.parametrize("radii,bound", [((1.0, 3.0), 1e-5), ((1.0, 1.0), 2 * 2.0 ** -11)])
def test_high_order_neighbours_of_unequal_radii(radii, bound):
    """Two spheres of order 12 at 1.55 radius sums.  Radii 1:3: the ratio that bounds
    the truncation is that of equal spheres at 1.37, so they stay on their own grids
    (FP32 sums).  Equal radii: the level of order 10, truncating less than 2^-11 on
    each side."""
    pos = np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 1.55 * sum(radii)]])
    quat = S.configs.Stream(2).quaternions(2)
    op = S.SphereSTKSHOperator(pos, np.array(radii), quat, np.array([12, 12], dtype=np.int32), 0.5, 0.0, 1.0, 1.0)
    x = density(op, 6)
    assert op.n_near_pairs == 0
    assert rel(op.apply_coarse(x), op.apply(x)) < bound
