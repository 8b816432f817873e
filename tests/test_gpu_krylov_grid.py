"""GMRES at the edges of its kernels' grid: fewer entries than a block's 512 threads, a ragged last block, and more than the
256 blocks take twice; restarts below, at and above the 8 basis vectors that a row of blocks takes, and the largest.
Explicit steps with the consistent mass solved by GMRES to 1e-10, against the oracle's: 1e-11 on the state, as in
test_gpu_ts.py (the update is a small part of it).  A solver reaches that solution with wrong sums too: the reductions
themselves are compared in test_gpu_reductions.py."""
import sys

import numpy as np
import pytest

import pyoracle as O
from pyhonee import mesh as M
from pyhonee import problems as PR
from pyhonee import ts as TS
from pyhonee.driver import NewtonianProblem, context_from_dict

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,restarts", [((3, 2, 2), (1, 7, 8, 9, 31)), ((5, 5, 5), (8, 16, 17)), ((38, 38, 37), (9,))])
def test_mass_solve(shape, restarts):
    L, dt = 2 * np.pi, 5e-3
    mesh, tab = M.box_mesh(shape, 1, lengths=(L, L, L), perturb=0.1, seed=3), M.tabulate(1, 0)
    d = PR.tgv_context_dict(state_var=0, stabilization=0, implicit=False, dt=dt, tau=PR.default_tau(1))
    rng = np.random.default_rng(3)
    Y = PR.nodal_field(mesh, lambda x: PR.taylor_green_prim(x))
    Y[:, 1:4] += 1e-3 * rng.uniform(-1, 1, Y[:, 1:4].shape)
    q0 = PR.q_from_prim(PR.TGV_GAS, Y, 0).ravel()
    om = O.Mesh(mesh, tab)
    A, b, cc = TS.tableau(TS.RK_EULER, 1)
    ref, _, _ = O.rk(om, O.newt_from_dict(d), om.setup_qdata(), q0, dt, 1, A, b, cc, t0=0.0, gmres=True, rowsum=False, rtol=1e-10)
    for restart in restarts:
        print(f"krylov grid shape={shape} restart={restart}", flush=True)
        sys.stdout.flush()
        prob = NewtonianProblem(mesh, tab, context_from_dict(d), 0)
        ts = TS.TimeStepper(prob, TS.default_options(type=TS.TS_RK, rk_type=TS.RK_EULER, dt=dt, mass_gmres=1, mass_jacobi_rowsum=0,
                                                      mass_rtol=1e-10, mass_restart=restart, mass_max_it=500))
        ts.set_solution(q0, 0.0)
        ts.step(1)
        q, st = ts.solution(), ts.stats()
        ts.close()
        prob.close()
        assert st["mass_krylov_its"] > 0
        e = np.linalg.norm(q - ref) / np.linalg.norm(ref)
        assert e < 1e-11, (restart, e)
