"""Transforms and near evaluation at the edges of their tiles: 16 spheres per
tile, 16 points or 48 coefficients per row block, 128 targets per near item,
orders up to the largest supported, mixed in one suspension."""
import os
import sys

import numpy as np
import pytest

from conftest import ROOT

sys.path.insert(0, os.path.join(ROOT, "oracle"))
pyoracle = pytest.importorskip("pyoracle")
S = pytest.importorskip("spheresimulator_amd")

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def line(n, gap, seed):
    """n spheres on a helix of wide turns, neighbours `gap` radii apart, others far."""
    r = np.random.default_rng(seed)
    rad = 0.7 + 0.6 * r.random(n)
    z = np.cumsum(rad) + np.concatenate([[0.0], np.cumsum(rad)[:-1]]) + gap * np.arange(n)
    pos = np.stack([0.3 * np.sin(z), 0.3 * np.cos(z), z], 1)
    return pos, rad, S.configs.Stream(seed).quaternions(n)


@pytest.mark.parametrize("n,orders", [(1, (20,)), (15, (1, 2, 3)), (16, (6,)), (17, (6,)), (33, (5, 7, 16)),
                                      (6, (13, 18, 20))])
def test_apply_and_projection_at_tile_edges(n, orders):
    """FP64 operator and projection against the oracle; sums of at most some
    thousand terms of size one: 1e-11 of the result, as for the other applies."""
    pos, rad, quat = line(n, 0.5, n)
    order = np.resize(np.array(orders, dtype=np.int32), n)
    c = (0.3, 0.7, 1.1, 0.9)
    op = S.SphereSTKSHOperator(pos, rad, quat, order, *c)
    ref = pyoracle.Operator(pos, rad, quat, order, *c)
    assert n == 1 or op.n_near_pairs > 0
    x = np.random.default_rng(n).standard_normal(op.n_dof)
    assert rel(op.apply(x), ref.apply(x)) < 1e-11
    y = x.copy()
    op.projectNullSpace(y)
    z = y.copy()
    op.projectNullSpace(z)
    assert rel(z, y) < 1e-11  # a projection
    assert rel(y, ref.project(x)) < 1e-11


@pytest.mark.parametrize("n,orders", [(17, (8,)), (33, (12,)), (40, (6, 10, 16))])
def test_multi_level_operators_at_tile_edges(n, orders):
    """Both multi-level operators on smooth densities of spheres far apart, where
    all pairs but the next ones go through levels: the bounds of the operator
    tests on random packings (outer 2e-9, coarse 5e-2) and for the inner one the
    5e-5 up to which two refinement steps reach 1e-8."""
    pos, rad, quat = line(n, 4.0, n + 100)
    order = np.resize(np.array(orders, dtype=np.int32), n)
    op = S.SphereSTKSHOperator(pos, rad, quat, order, 0.5, 0.0, 1.0, 1.0)
    x = np.random.default_rng(n).standard_normal(op.n_dof)
    op.projectNullSpace(x)
    y = op.apply(x)
    assert rel(op.apply_outer(x), y) < 2e-9
    assert rel(op.apply_inner(x), y) < 5e-5
    assert rel(op.apply_coarse(x), y) < 5e-2


@pytest.mark.parametrize("n,orders", [(17, (11,)), (18, (10, 11)), (20, (16, 12, 8)), (5, (20,))])
def test_coarse_operator_with_next_neighbours_on_a_level(n, orders):
    """Neighbours between 1.5 and 2 (R_s + R_t), which orders above 10 sum on a
    level of order 10: its truncation there is at most 2^-11, order 5's behind it
    1.1e-3; ten times the larger for the handful of degrees at the cut."""
    pos, rad, quat = line(n, 1.5, n + 200)
    order = np.resize(np.array(orders, dtype=np.int32), n)
    op = S.SphereSTKSHOperator(pos, rad, quat, order, 0.5, 0.0, 1.0, 1.0)
    x = np.random.default_rng(n).standard_normal(op.n_dof)
    op.projectNullSpace(x)
    assert rel(op.apply_coarse(x), op.apply(x)) < 1.1e-2
