"""The diagonals into vectors that hold other values, twice, for both scatters.  The point blocks of the two-pass scatter and the
Jacobi diagonal of its larger meshes go through the E-vector, whose gather overwrites the output where its rows cover it; the
others add to a cleared vector.  Tolerances of test_gpu_parity.py (the same sums in another order)."""
import sys

import numpy as np
import pytest

import pyoracle as O
from helpers import make_case, oracle_setup, product_context, rel_err
from pyhonee.driver import NewtonianProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,shape", [(1, (1, 1, 1)), (1, (7, 3, 2)), (2, (3, 3, 1)), (3, (2, 3, 2)), (4, (1, 2, 1))])
@pytest.mark.parametrize("scatter", ["twopass", "atomic"])
def test_diagonals_overwrite(degree, shape, scatter):
    print(f"diagonal scatter degree={degree} shape={shape} {scatter}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), perturb=0.1, state_var=1, stabilization=2, seed=21)
    om, oc, qd = oracle_setup(case)
    _, jac = O.ifunction(om, oc, qd, case["q"], case["qdot"])
    oc.ijacobian_time_shift = 90.0
    d_ref, pb_ref = O.ijacobian_diagonal(om, oc, qd, jac), O.ijacobian_point_block_diagonal(om, oc, qd, jac)
    prob = NewtonianProblem(case["mesh"], case["tab"], product_context(case), 1, f"/gpu/hip/mi355x:scatter={scatter}")
    g = np.zeros_like(case["q"])
    prob.ifunction(case["q"], case["qdot"], g)
    d, pb = np.full_like(case["q"], 7.0), np.full((om.nnodes, 5, 5), -3.0)
    for _ in range(2):
        prob.ijacobian_diagonal(d, 90.0)
        prob.ijacobian_point_block_diagonal(pb, 90.0)
        for x, ref in ((d, d_ref), (pb, pb_ref)):
            e2, emax = rel_err(x, np.reshape(ref, x.shape))
            assert e2 < 1e-12 and emax < 1e-11, (e2, emax)
    prob.close()


@pytest.mark.parametrize("degree,shape", [(1, (30, 30, 28)), (2, (16, 16, 15)), (3, (12, 12, 11)), (4, (16, 10, 10))])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_jacobi_diagonal_of_larger_meshes(degree, shape, precision):
    """Just above the sizes from which the two-pass scatter's Jacobi diagonal goes through the E-vector, against the atomic one."""
    print(f"diagonal scatter degree={degree} shape={shape} {precision}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), perturb=0.1, state_var=1, stabilization=2, seed=22)
    d = {}
    for scatter in ("twopass", "atomic"):
        prob = NewtonianProblem(case["mesh"], case["tab"], product_context(case), 1,
                                f"/gpu/hip/mi355x:scatter={scatter}:jacobian_precision={precision}")
        prob.ifunction(case["q"], case["qdot"], np.zeros_like(case["q"]))
        d[scatter] = [np.full_like(case["q"], 7.0) for _ in range(2)]
        for x in d[scatter]:
            prob.ijacobian_diagonal(x, 90.0)
        prob.close()
    e2, emax = rel_err(d["twopass"][0], d["atomic"][0])
    assert e2 < 1e-12 and emax < 1e-11, (e2, emax)
    assert (d["twopass"][0] == d["twopass"][1]).all()
