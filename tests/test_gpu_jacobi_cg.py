"""The conjugate gradients with the scalars on the device, against the oracle's solve of the filter system: fewer entries
than one block, a few blocks with a ragged last one, and more entries than one pass of the largest grid.  Both stop at
rtol = 1e-10 in the natural norm, from which the two solutions may differ: 1e-9 relative, as for the solve in general."""
import sys

import pytest

import pyoracle as O
from helpers import make_case, oracle_setup, product_context, rel_err
from pyhonee.driver import NewtonianProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,shape", [(1, (1, 1, 1)), (1, (3, 3, 2)), (2, (3, 3, 3)), (1, (29, 29, 28))])
def test_solve_at_grid_edges(degree, shape):
    print(f"jacobi cg degree={degree} shape={shape}", flush=True)
    sys.stdout.flush()
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), perturb=0.1, state_var=1, stabilization=0, seed=7)
    om, oc, qd = oracle_setup(case)
    prob = NewtonianProblem(case["mesh"], case["tab"], product_context(case), 1)
    prob.setup_diff_filter(grid_based_width=True, width_scaling=(1.5, 0.7, 1.0))
    runs = [prob.diff_filter_apply(case["q"]) for _ in range(2)]
    prob.close()
    f = O.diff_filter(grid_based_width=True, width_scaling=(1.5, 0.7, 1.0), damping=0, friction_length=0.0)
    ref, its = O.diff_filter_solve(om, f, qd, O.anisotropy_collocate(om, qd), 11, O.diff_filter_rhs(om, oc, qd, case["q"]))
    for x, n in runs:
        assert abs(n - its) <= 1, (n, its)
        e2, emax = rel_err(x, ref)
        assert e2 < 1e-9 and emax < 1e-8, (e2, emax)
    assert (runs[0][0] == runs[1][0]).all() and runs[0][1] == runs[1][1]
