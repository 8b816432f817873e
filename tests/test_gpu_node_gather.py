"""The tiled gather of the element-ordered E-vector where its tiles take another form: a row with more contributions than a
tile of small meshes aims at (100 elements share a node), one with more than a tile can hold (648), and the FP32
contributions of the mixed-precision Jacobian in the same tiles.  Element counts without shared rows of that size are in the
parity tests.  The sums are the oracle's in another order: tolerances of test_gpu_parity.py, and for FP32 of its apply."""
import sys

import numpy as np
import pytest

import pyoracle as O
from helpers import make_case, rel_err
from pyhonee import mesh as M
from pyhonee.driver import NewtonianProblem, context_from_dict

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree", [1, 2])
@pytest.mark.parametrize("shape", [(5, 5, 4), (9, 9, 8)])
@pytest.mark.parametrize("fp32", [False, True])
def test_rows_of_many_contributions(degree, shape, fp32):
    print(f"node gather degree={degree} shape={shape} fp32={fp32}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), seed=11 + degree)
    # the last node of every element becomes node 0; the nodes that no element names any more keep their rows
    offsets = np.ascontiguousarray(case["mesh"].offsets).reshape(-1, (degree + 1) ** 3)
    offsets[:, -1] = offsets[0, 0]
    case["mesh"].offsets = offsets.reshape(np.shape(case["mesh"].offsets))
    tab = M.tabulate(degree, 0)
    om, oc = O.Mesh(case["mesh"], tab), O.newt_from_dict(case["ctx"])
    qd = om.setup_qdata()
    v_ref, jac_ref = O.ifunction(om, oc, qd, case["q"], case["qdot"])
    dq = case["rng"].uniform(-1e-3, 1e-3, case["q"].shape)
    oc.ijacobian_time_shift = 100.0
    j_ref = O.ijacobian(om, oc, qd, jac_ref, dq)
    prob = NewtonianProblem(case["mesh"], tab, context_from_dict(case["ctx"]), 1,
                            "/gpu/hip/mi355x:jacobian_precision=fp32" if fp32 else "/gpu/hip/mi355x")
    g, v = np.zeros_like(case["q"]), np.zeros_like(case["q"])
    prob.ifunction(case["q"], case["qdot"], g)
    prob.ijacobian(dq, v, 100.0)
    prob.close()
    assert rel_err(g, v_ref)[0] < 1e-12 and rel_err(g, v_ref)[1] < 1e-11, rel_err(g, v_ref)
    tol = 2e-5 if fp32 else 1e-12
    assert rel_err(v, j_ref)[0] < tol, rel_err(v, j_ref)


@pytest.mark.parametrize("degree,shape", [(1, (3, 2, 2)), (1, (16, 8, 8)), (1, (41, 5, 5)), (2, (7, 7, 6)), (2, (9, 9, 8)), (3, (9, 7, 5))])
def test_shuffled_node_numbers(degree, shape):
    """The tables of the gather as the host lays them out (up to 8192 element nodes, the second case) and as the device does (the
    third and on), for nodes in no order along the elements; the second apply runs on the tables of the first."""
    print(f"node gather shuffled degree={degree} shape={shape}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, True, False), seed=5 + degree)
    number = case["rng"].permutation(case["mesh"].nnodes).astype(np.int32)
    case["mesh"].offsets = np.ascontiguousarray(number[np.asarray(case["mesh"].offsets)])
    tab = M.tabulate(degree, 0)
    om, oc = O.Mesh(case["mesh"], tab), O.newt_from_dict(case["ctx"])
    v_ref, _ = O.ifunction(om, oc, om.setup_qdata(), case["q"], case["qdot"])
    prob = NewtonianProblem(case["mesh"], tab, context_from_dict(case["ctx"]), 1)
    g = [np.full_like(case["q"], 3.0) for _ in range(2)]
    for x in g:
        prob.ifunction(case["q"], case["qdot"], x)
    prob.close()
    assert rel_err(g[0], v_ref)[0] < 1e-12 and rel_err(g[0], v_ref)[1] < 1e-11, rel_err(g[0], v_ref)
    assert (g[0] == g[1]).all()
