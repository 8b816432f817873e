"""Runge-Kutta stages with the point-diagonal mass solve in the stage's kernel: every scheme (zero coefficients, derivatives
that a later stage needs or not), more stages than the kernel takes, and lengths below a block, with a ragged last block and
above one pass of the last stage's grid.  Against the oracle's steps: 1e-11 on the state, as in test_gpu_ts.py."""
import sys

import numpy as np
import pytest

import pyoracle as O
from pyhonee import mesh as M
from pyhonee import problems as PR
from pyhonee import ts as TS
from pyhonee.driver import NewtonianProblem, context_from_dict

pytestmark = pytest.mark.gpu


SCHEMES = [(TS.RK_EULER, 1), (TS.RK_4, 4), (TS.RK_5F, 6), (TS.RK_SSP33, 3), (TS.RK_SSP_S3, 4), (TS.RK_SSP_S3, 9)]


@pytest.mark.parametrize("rk_type,stages,shape", [(*s, n) for s in SCHEMES for n in ((3, 2, 2), (7, 6, 5))] + [(TS.RK_SSP33, 3, (60, 60, 59))])
def test_lumped_steps(rk_type, stages, shape):
    print(f"rk stage rk={rk_type} stages={stages} shape={shape}", flush=True)
    sys.stdout.flush()
    L, dt, steps = 2 * np.pi, 5e-3, 2
    mesh, tab = M.box_mesh(shape, 1, lengths=(L, L, L), perturb=0.1, seed=4), M.tabulate(1, 0)
    d = PR.tgv_context_dict(state_var=0, stabilization=0, implicit=False, dt=dt, tau=PR.default_tau(1))
    q0 = PR.q_from_prim(PR.TGV_GAS, PR.nodal_field(mesh, lambda x: PR.taylor_green_prim(x)), 0).ravel()
    om = O.Mesh(mesh, tab)
    A, b, cc = TS.tableau(rk_type, stages)
    ref, _, _ = O.rk(om, O.newt_from_dict(d), om.setup_qdata(), q0, dt, steps, A, b, cc, t0=0.0, gmres=False, rowsum=True, rtol=1e-10)
    prob = NewtonianProblem(mesh, tab, context_from_dict(d), 0)
    ts = TS.TimeStepper(prob, TS.default_options(type=TS.TS_RK, rk_type=rk_type, ssp_stages=stages, dt=dt, mass_gmres=0, mass_jacobi_rowsum=1))
    ts.set_solution(q0, 0.0)
    ts.step(steps)
    q, st = ts.solution(), ts.stats()
    ts.close()
    prob.close()
    assert st["rhs_evals"] == steps * len(b)
    e = np.linalg.norm(q - ref) / np.linalg.norm(ref)
    assert e < 1e-11, e
