"""GMRES vector kernels on a suspension of so many unknowns that its chunk
partials are added up by launches of their own (more than 1024 chunks of 4096)."""
import numpy as np
import pytest

S = pytest.importorskip("spheresimulator_amd")

pytestmark = pytest.mark.gpu


def test_gram_schmidt_forms_agree_beyond_the_sums_in_blocks():
    """4200 spheres p=12, 4.26e6 unknowns, mixed form: restart 64 takes modified
    Gram-Schmidt step by step, restart 60 classical Gram-Schmidt twice.  Both build the
    same Krylov spaces, so the iterations agree (but for one at a tolerance's edge in
    each of the three refinement steps) and the velocities to ten times the solves'
    tolerance of 1e-8."""
    n = 4200
    c = S.configs.make_suspension(n, 12, 31, vf=0.05, min_gap=0.2)
    out = []
    for restart in (60, 64):
        m = S.SphereSTKMobMat(c["pos"], c["radius"], c["quat"], c["order"], precision=S.PREC_MIXED,
                              params=S.solver_params(restart=restart))
        assert m.n_dof > 1024 * 4096
        v, info = m.solveMob(c["force"])
        assert info["converged"] and info["relres"] < 1e-8
        out.append((v, info["iters"]))
        del m
    assert abs(out[0][1] - out[1][1]) <= 3
    assert np.linalg.norm(out[0][0] - out[1][0]) < 1e-7 * np.linalg.norm(out[0][0])
