"""Operator applies that the iterative solvers launch before the host has seen whether they converge: all of them are used.  The
launches are those that the operator's timer counts, against the applies that the solve reports or needs (one an iteration)."""
import sys

import numpy as np
import pytest

from helpers import make_case, product_context
from pyhonee import mesh as M
from pyhonee import problems as PR
from pyhonee import ts as TS
from pyhonee.driver import NewtonianProblem, context_from_dict

pytestmark = pytest.mark.gpu


def _launches(prob, name):
    return sum(n for k, (n, _) in prob.kernel_times().items() if k == name)


def _problem(shape, degree, implicit):
    L = 2 * np.pi
    mesh, tab = M.box_mesh(shape, degree, lengths=(L, L, L), perturb=0.1, seed=4), M.tabulate(degree, 0)
    var = 1 if implicit else 0
    d = PR.tgv_context_dict(state_var=var, stabilization=2 if implicit else 0, implicit=implicit, dt=2e-3, tau=PR.default_tau(degree))
    q0 = PR.q_from_prim(PR.TGV_GAS, PR.nodal_field(mesh, lambda x: PR.taylor_green_prim(x)), var).ravel()
    return NewtonianProblem(mesh, tab, context_from_dict(d), var), q0


@pytest.mark.parametrize("kind,shape,degree", [("jacobian", (4, 4, 4), 3), ("jacobian", (5, 4, 3), 2), ("mass", (4, 4, 4), 3), ("mass", (6, 5, 4), 2)])
def test_gmres(kind, shape, degree):
    print(f"apply ahead {kind} shape={shape} degree={degree}", flush=True)
    sys.stdout.flush()
    prob, q0 = _problem(shape, degree, kind == "jacobian")
    if kind == "jacobian":
        o = TS.default_options(type=TS.TS_BDF, dt=2e-3, ksp_pc=TS.PC_PBJACOBI)
    else:
        o = TS.default_options(type=TS.TS_RK, rk_type=TS.RK_SSP33, dt=1e-3, mass_gmres=1, mass_jacobi_rowsum=0, mass_rtol=1e-6)
    ts = TS.TimeStepper(prob, o)
    ts.set_solution(q0, 0.0)
    ts.step(1)
    before = ts.stats()
    prob.set_timing(True)
    prob.reset_times()
    ts.step(2)
    launched, st = prob.kernel_times(), ts.stats()
    prob.set_timing(False)
    ts.close()
    prob.close()
    name = next(k for k in launched if k.startswith("ijacobian" if kind == "jacobian" else "mass") and "diagonal" not in k)
    used = st[f"{kind}_applies"] - before[f"{kind}_applies"]
    assert used > 4
    assert launched[name][0] == used, launched


@pytest.mark.parametrize("degree,shape", [(1, (4, 4, 3)), (2, (4, 3, 3)), (3, (2, 2, 3))])
def test_filter_cg(degree, shape):
    print(f"apply ahead filter degree={degree} shape={shape}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), perturb=0.1, state_var=1, stabilization=0, seed=7)
    prob = NewtonianProblem(case["mesh"], case["tab"], product_context(case), 1)
    prob.setup_diff_filter(grid_based_width=True)
    prob.diff_filter_apply(case["q"])
    prob.set_timing(True)
    prob.reset_times()
    _, its = prob.diff_filter_apply(case["q"])
    launched = prob.kernel_times()
    prob.set_timing(False)
    prob.close()
    assert its > 4 and launched["diff_filter_lhs"][0] == its, launched
