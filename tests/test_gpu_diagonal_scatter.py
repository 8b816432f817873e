"""The diagonals through the E-vector, whose gather overwrites the output where its rows cover it: into vectors that hold
other values, twice, for both scatters (the atomic one adds to a cleared vector), from one element up.  Tolerances of
test_gpu_parity.py (the same sums in another order)."""
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
