"""The filter operator for 1, 5 and 6 components as a program that registers the reference's QFunctions makes it
(DifferentialFilter_LHS_1, and the composite of _5 and _6 on the interleaved 11-component field, src/differential_filter.c:90-149),
with both scatters, and both scatters of the framework's own 11-component operator and right-hand side: element counts around a
block's 8 (Q = 2), 2 (Q = 3) and 1 elements and a wave's 5.  Tolerances of test_gpu_filter.py."""
import ctypes as ct
import sys

import numpy as np
import pytest

import pyoracle as O
from ceed_objects import COPY_VALUES, GRAD, INTERP, NONE, CeedObjects
from helpers import make_case, oracle_setup, product_context, rel_err
from pyhonee.driver import CEED_MEM_HOST, NewtonianContext, NewtonianProblem

pytestmark = pytest.mark.gpu

FILTER = dict(grid_based_width=True, width_scaling=(1.5, 0.7, 1.0))


class FilterContext(ct.Structure):
    _fields_ = [("grid_based_width", ct.c_bool), ("width_scaling", ct.c_double * 3), ("kernel_scaling", ct.c_double), ("friction_length", ct.c_double),
                ("damping_function", ct.c_int), ("damping_constant", ct.c_double), ("newt_ctx", NewtonianContext)]


class FilterLHS(CeedObjects):
    """Composite of DifferentialFilter_LHS_N over the component ranges [(offset, N), ...] of an 11-component field."""

    def __init__(self, prob, aniso, parts):
        super().__init__(prob)
        mesh, tab, ceed = prob.mesh, prob.tab, self.ceed
        self.n = 11 * mesh.nnodes
        x, bx = self._restriction(mesh.nelem, 8, 3, 3 * prob.m.nxnodes, 3 * np.asarray(mesh.xoffsets)), self._basis(3, 2, prob._keep["Bx"], prob._keep["Dx"])
        ctx = FilterContext(True, (ct.c_double * 3)(*FILTER["width_scaling"]), 0.1, 0.0, 0, 25.0, prob.ctx)
        qctx = self._made("CeedQFunctionContextCreate", ceed)
        self._call("CeedQFunctionContextSetData", qctx, CEED_MEM_HOST, COPY_VALUES, ct.c_size_t(ct.sizeof(ctx)), ct.byref(ctx))
        active, no_basis = self._pointer("CEED_VECTOR_ACTIVE"), self._pointer("CEED_BASIS_NONE")
        passive = {"anisotropy tensor": (self.strided(7), no_basis, self.vector(aniso)), "x": (x, bx, self.vector(prob._keep["xcoord"])),
                   "qdata": (self.strided(10), no_basis, self.vector(prob.qdata()))}
        self.op = self._made("CeedOperatorCreateComposite", ceed)
        for offset, N in parts:
            f = (self._restriction(mesh.nelem, tab.P ** 3, N, self.n, 11 * np.asarray(mesh.offsets) + offset),
                 self._basis(N, tab.P, prob._keep["B"], prob._keep["D"]), active)
            sub = self.operator(f"qfunctions/differential_filter.h:DifferentialFilter_LHS_{N}", qctx,
                                [("q", N, INTERP), ("Grad_q", 3 * N, GRAD), ("anisotropy tensor", 7, NONE), ("x", 3, INTERP), ("qdata", 10, NONE)],
                                [("v", N, INTERP), ("Grad_v", 3 * N, GRAD)], {"q": f, "Grad_q": f, **passive, "v": f, "Grad_v": f})
            self._call("CeedOperatorCompositeAddSub", self.op, sub)

    def apply(self, vin, vout):
        self._call("CeedOperatorApply", self.op, vin, vout, None)

    def diagonal(self, vout):
        self._call("CeedOperatorLinearAssembleDiagonal", self.op, vout, None)


def _case(degree, shape, scatter):
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), perturb=0.1, state_var=1, stabilization=0, seed=40 + degree)
    om, oc, qd = oracle_setup(case)
    prob = NewtonianProblem(case["mesh"], case["tab"], product_context(case), 1, f"/gpu/hip/mi355x:scatter={scatter}")
    return case, om, oc, qd, prob, O.anisotropy_collocate(om, qd), O.diff_filter(**FILTER, damping=0, friction_length=0.0)


SIZES = [(1, (1, 1, 1)), (1, (7, 1, 1)), (1, (3, 3, 1)), (2, (1, 1, 1)), (2, (3, 1, 1)), (2, (3, 2, 1)), (2, (11, 1, 1)), (3, (1, 1, 1)), (3, (2, 3, 1)),
         (4, (1, 1, 1)), (4, (2, 1, 2))]


@pytest.mark.parametrize("degree,shape", SIZES)
@pytest.mark.parametrize("scatter", ["twopass", "atomic"])
@pytest.mark.parametrize("parts", [((0, 5), (5, 6)), ((3, 1),), ((5, 6), (2, 1))])
def test_operator_of_components(degree, shape, scatter, parts):
    print(f"filter components degree={degree} shape={shape} {scatter} {parts}", flush=True)
    sys.stdout.flush()
    case, om, _, qd, prob, acol, f = _case(degree, shape, scatter)
    u = case["rng"].uniform(-1, 1, (case["mesh"].nnodes, 11))
    lhs = FilterLHS(prob, acol, parts)
    vin, vout = lhs.vector(u), lhs.vector(np.full(u.shape, 7.0))
    mine = np.zeros(11, dtype=bool)
    for offset, N in parts:
        mine[offset:offset + N] = True
    ref = O.diff_filter_lhs(om, f, qd, acol, 11, u).reshape(-1, 11) * mine
    dref = O.diff_filter_lhs_diagonal(om, f, qd, acol, 11).reshape(-1, 11) * mine
    for _ in range(2):
        lhs.apply(vin, vout)
        e2, emax = rel_err(lhs.read(vout, lhs.n).reshape(-1, 11), ref)
        assert e2 < 1e-12 and emax < 1e-11, (e2, emax)
    lhs.diagonal(vout)
    e2, emax = rel_err(lhs.read(vout, lhs.n).reshape(-1, 11), dref)
    assert e2 < 1e-12 and emax < 1e-11, (e2, emax)
    prob.close()


@pytest.mark.parametrize("degree,shape", SIZES)
@pytest.mark.parametrize("scatter", ["twopass", "atomic"])
def test_framework_operators(degree, shape, scatter):
    print(f"filter components 11 degree={degree} shape={shape} {scatter}", flush=True)
    sys.stdout.flush()
    case, om, oc, qd, prob, acol, f = _case(degree, shape, scatter)
    prob.setup_diff_filter(**FILTER)
    u = case["rng"].uniform(-1, 1, (case["mesh"].nnodes, 11))
    v, d = prob.diff_filter_lhs(u)
    rhs = prob.diff_filter_rhs(case["q"])
    prob.close()
    for x, ref in ((v, O.diff_filter_lhs(om, f, qd, acol, 11, u)), (d, O.diff_filter_lhs_diagonal(om, f, qd, acol, 11)),
                   (rhs, O.diff_filter_rhs(om, oc, qd, case["q"]))):
        e2, emax = rel_err(x, np.reshape(ref, x.shape))
        assert e2 < 1e-12 and emax < 1e-11, (e2, emax)
