"""The line-per-thread basis stage at the edges of its blocks, against the oracle: element counts around the 8 (Q = 2) and 2
(Q = 3) elements of a block, one element, and (P, Q) pairs whose lines fill a round exactly, leave lanes over, or leave a
whole wave without lines (Q = 6).  Tolerances are those of test_gpu_parity.py (rounding of the same sums in another order)."""
import sys

import numpy as np
import pytest

import pyoracle as O
from helpers import make_case, rel_err
from pyhonee import mesh as M
from pyhonee.driver import NewtonianProblem, context_from_dict

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,q_extra", [(1, 0), (1, 1), (1, 2), (2, 0), (2, 1), (2, 2), (3, 1), (3, 2), (4, 0)])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 1, 1), (7, 1, 1), (3, 3, 1), (17, 1, 1)])
@pytest.mark.parametrize("scatter", ["twopass", "atomic"])
def test_residual_and_jacobian_at_block_edges(degree, q_extra, shape, scatter):
    print(f"line stage degree={degree} q_extra={q_extra} shape={shape} {scatter}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), seed=3 + degree)
    tab = M.tabulate(degree, q_extra)
    om, oc = O.Mesh(case["mesh"], tab), O.newt_from_dict(case["ctx"])
    qd = om.setup_qdata()
    v_ref, jac_ref = O.ifunction(om, oc, qd, case["q"], case["qdot"])
    dq = case["rng"].uniform(-1e-3, 1e-3, case["q"].shape)
    oc.ijacobian_time_shift = 100.0
    j_ref = O.ijacobian(om, oc, qd, jac_ref, dq)
    prob = NewtonianProblem(case["mesh"], tab, context_from_dict(case["ctx"]), 1, f"/gpu/hip/mi355x:scatter={scatter}")
    g, v = np.zeros_like(case["q"]), np.zeros_like(case["q"])
    prob.ifunction(case["q"], case["qdot"], g)
    prob.ijacobian(dq, v, 100.0)
    prob.close()
    assert rel_err(g, v_ref)[0] < 1e-12 and rel_err(g, v_ref)[1] < 1e-11, rel_err(g, v_ref)
    assert rel_err(v, j_ref)[0] < 1e-12 and rel_err(v, j_ref)[1] < 1e-11, rel_err(v, j_ref)


@pytest.mark.parametrize("degree", [1, 2, 3, 4])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 1, 1), (3, 3, 1)])
def test_filter_operator_at_block_edges(degree, shape):
    """The filter operator: its right-hand side runs the same stage with 11 outputs, its left-hand side with 6 components at a time at
    degree 4 (degrees 1 and 2 have a kernel of a lane per component, degree 3 the 4 x 4 x 4 element's stages)."""
    print(f"line stage filter degree={degree} shape={shape}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), seed=13 + degree)
    prob = NewtonianProblem(case["mesh"], case["tab"], context_from_dict(case["ctx"]), 1)
    prob.setup_diff_filter(grid_based_width=True)
    om = O.Mesh(case["mesh"], case["tab"])
    qd = om.setup_qdata()
    u = case["rng"].uniform(-1, 1, (case["mesh"].nnodes, 11))
    v, diag = prob.diff_filter_lhs(u)
    rhs = prob.diff_filter_rhs(case["q"])
    prob.close()
    f, acol = O.diff_filter(grid_based_width=True), O.anisotropy_collocate(om, qd)
    v_ref = O.diff_filter_lhs(om, f, qd, acol, 11, u)
    d_ref = O.diff_filter_lhs_diagonal(om, f, qd, acol, 11)
    rhs_ref = O.diff_filter_rhs(om, O.newt_from_dict(case["ctx"]), qd, case["q"])
    for x, ref in ((v, v_ref), (diag, d_ref), (rhs, rhs_ref)):
        assert rel_err(x, ref)[0] < 1e-12, rel_err(x, ref)
