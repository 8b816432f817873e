"""The backend's host code on a HIP runtime of host memory that counts kernels instead of running them (fake_hip.c): what a first
apply uploads, which route a diagonal takes, and that a failed allocation is an error and leaves the objects usable."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as ct, sys
import numpy as np
from helpers import make_case, product_context
from pyhonee import mesh as M
from pyhonee.driver import NewtonianProblem
hip = ct.CDLL(None)
hip.fake_h2d_bytes.restype = hip.fake_dev_bytes.restype = ct.c_longlong
hip.fake_launches.restype = ct.c_long
hip.fake_launches.argtypes = [ct.c_char_p]
hip.fake_fail_malloc.argtypes = hip.fake_fail_host_malloc.argtypes = [ct.c_long]
def problem(shape=(4, 4, 4), degree=2, q_extra=0, resource="/gpu/hip/mi355x"):
    case = make_case(shape=shape, degree=degree, periodic=(False, False, False), state_var=1, stabilization=2, seed=7)
    return case, NewtonianProblem(case["mesh"], M.tabulate(degree, q_extra), product_context(case), 1, resource)
def uploaded(f):
    before = hip.fake_h2d_bytes()
    f()
    return hip.fake_h2d_bytes() - before
def refused(f):
    try:
        f()
    except RuntimeError as e:
        return str(e)
    raise AssertionError("not refused")
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    lib = tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(lib), os.path.join(HERE, "fake_hip.c")], check=True)
    return str(lib)


def _run(fake, body):
    preload = " ".join(p for p in (fake, os.environ.get("LD_PRELOAD")) if p)
    env = dict(os.environ, LD_PRELOAD=preload, PYTHONPATH=os.pathsep.join(sys.path))
    r = subprocess.run([sys.executable, "-c", PRELUDE + body], env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-500:], r.stderr[-2000:])


def test_first_apply_uploads_the_map_alone(fake):
    """The offsets, the rows with their element nodes, a few words a tile and the basis tables; the rest of the gather's tables is
    laid out by the device.  Operators that do not gather with tiles have none."""
    _run(fake, """
case, prob = problem((8, 8, 8))
n, rows = case["mesh"].offsets.size, case["mesh"].nnodes
g = np.zeros_like(case["q"])
apply = lambda: prob.ifunction(case["q"], case["qdot"], g)
first, again = uploaded(apply), uploaded(apply)
assert first - again <= 4 * (2 * n + 2 * rows + 1) + 4 * (n // 32) + 1024, (first, again, n, rows)
assert hip.fake_launches(b"k_layout_tiles") == 1
prob.setup_diff_filter(grid_based_width=True)
filt = lambda: prob.diff_filter_lhs(np.zeros((rows, 11)))
first, again = uploaded(filt), uploaded(filt)
assert hip.fake_launches(b"k_layout_tiles") == 1
""")


def test_conjugate_gradients_without_host_memory(fake):
    """The solve allocates device and mapped host memory at its first call; without the latter it is an error, also again."""
    _run(fake, """
case, prob = problem()
prob.setup_diff_filter(grid_based_width=True)
hip.fake_fail_host_malloc(0)
assert "OutOfMemory" in refused(lambda: prob.diff_filter_apply(case["q"]))
hip.fake_fail_host_malloc(0)
assert "OutOfMemory" in refused(lambda: prob.diff_filter_apply(case["q"]))
assert "not published" in refused(lambda: prob.diff_filter_apply(case["q"]))  # the kernels do not run here
""")


def test_workspace_that_could_not_grow(fake):
    """The E-vector's workspace is freed before a larger one is allocated; without that one, the next smaller apply allocates its own
    (with none the kernel would add to an output that nothing has cleared)."""
    _run(fake, """
case, prob = problem()
g, pb = np.zeros_like(case["q"]), np.zeros((case["mesh"].nnodes, 5, 5))
apply = lambda: prob.ifunction(case["q"], case["qdot"], g)
apply()
assert hip.fake_launches(b"k_node_gather_tiles") == 1
hip.fake_fail_malloc(1)  # the point blocks' vector, then the workspace
assert "OutOfMemory" in refused(lambda: prob.ijacobian_point_block_diagonal(pb, 90.0))
apply()
assert hip.fake_launches(b"k_node_gather_tiles") == 2
""")


def test_first_apply_with_a_failed_allocation(fake):
    """Whichever allocation of a first apply fails (vectors, basis tables, maps, workspace), in the end all is there that a first apply
    allocates: later in the same apply, where its preparation is tried again, or in the next one, after an error."""
    _run(fake, """
def first_apply(fail):
    case, prob = problem((3, 2, 2))
    g, start, errors = np.zeros_like(case["q"]), hip.fake_dev_bytes(), 0
    hip.fake_fail_malloc(fail)
    try:
        prob.ifunction(case["q"], case["qdot"], g)
    except RuntimeError as e:
        assert "OutOfMemory" in str(e), e
        errors = 1
        prob.ifunction(case["q"], case["qdot"], g)
    hip.fake_fail_malloc(-1)
    return hip.fake_dev_bytes() - start, errors
needed, _ = first_apply(-1)
sizes, errors = zip(*[first_apply(k) for k in range(20)])
assert all(size == needed for size in sizes), (needed, sizes)
assert 0 < sum(errors) < 20, errors
""")


def test_training_buffers_that_could_not_grow(fake):
    """The network's staging, partials and sample order are freed before larger ones are allocated; without those, the smaller batches
    that ran before get buffers of their own, and nothing is freed twice."""
    _run(fake, """
from pyhonee import train as TR
def arrays(n):
    return np.ones((n, 6), dtype=np.float32), np.ones((n, 6), dtype=np.float32)
o, failures = TR.options(batch=64), 0
for k in range(6):
    mlp = TR.Mlp(seed=1)
    small, large = arrays(200), arrays(4000)
    mlp.train(*small, o), mlp.loss_grad(*small)
    for f in (lambda a: mlp.loss_grad(*a), lambda a: mlp.train(*a, o)):
        hip.fake_fail_malloc(k)
        try:
            f(large)
        except RuntimeError:
            failures += 1
        hip.fake_fail_malloc(-1)
        f(small)
        f(large)
    mlp.close()
assert failures > 3, failures
""")


@pytest.mark.parametrize("shape,degree,q_extra,scatter,gathered", [
    ((30, 30, 28), 1, 0, "twopass", 1), ((30, 30, 27), 1, 0, "twopass", 0), ((16, 16, 15), 2, 0, "twopass", 1), ((15, 15, 15), 2, 0, "twopass", 0),
    ((12, 12, 11), 3, 0, "twopass", 1), ((11, 11, 12), 3, 0, "twopass", 0), ((16, 10, 10), 4, 0, "twopass", 1), ((3, 2, 2), 3, 0, "twopass", 0),
    ((30, 30, 28), 1, 1, "twopass", 0), ((16, 16, 15), 2, 1, "twopass", 0), ((12, 12, 11), 3, 0, "atomic", 0)])
def test_route_of_the_jacobi_diagonal(fake, shape, degree, q_extra, scatter, gathered):
    """Through the E-vector, whose gather overwrites the output, where that is faster; else atomically into a cleared vector.  The
    point blocks have their own gather, which overwrites in the two-pass scatter."""
    _run(fake, f"""
case, prob = problem({shape}, {degree}, {q_extra}, "/gpu/hip/mi355x:scatter={scatter}")
g, pb = np.zeros_like(case["q"]), np.zeros((case["mesh"].nnodes, 5, 5))
prob.ifunction(case["q"], case["qdot"], g)
count = lambda name: hip.fake_launches(name)
before = count(b"k_node_gather_tiles"), count(b"k_fill")
prob.ijacobian_diagonal(g, 90.0)
assert count(b"k_node_gather_tiles") - before[0] == {gathered}
assert count(b"k_fill") - before[1] == 1 - {gathered}
before = count(b"k_node_gather_blocks"), count(b"k_fill")
prob.ijacobian_point_block_diagonal(pb, 90.0)
assert count(b"k_node_gather_blocks") - before[0] == 1
assert count(b"k_fill") - before[1] == {int(scatter == "atomic")}
""")


@pytest.mark.parametrize("shape,point_block", [((3, 2, 2), False), ((16, 16, 15), False), ((3, 2, 2), True)])
def test_allocation_free_apply_behind_a_diagonal(fake, shape, point_block):
    """An assembled diagonal prepares an operator for the allocation-free apply as an apply does, whichever route it took."""
    _run(fake, f"""
from ceed_objects import INTERP, NONE, CeedObjects
case, prob = problem({shape})
mesh, tab, c = case["mesh"], case["tab"], CeedObjects(prob)
r = c._restriction(mesh.nelem, tab.P ** 3, 5, 5 * mesh.nnodes, 5 * np.asarray(mesh.offsets))
f = (r, c._basis(5, tab.P, prob._keep["B"], prob._keep["D"]), c._pointer("CEED_VECTOR_ACTIVE"))
op = c.operator("qfunctions/mass.h:Mass_5", None, [("u", 5, INTERP), ("qdata", 10, NONE)], [("v", 5, INTERP)],
                {{"u": f, "qdata": (c.strided(10), c._pointer("CEED_BASIS_NONE"), c.vector(prob.qdata())), "v": f}})
v, w = c.vector(np.zeros(5 * mesh.nnodes)), c.vector(np.zeros(5 * mesh.nnodes))
d = c.vector(np.zeros(({25 if point_block else 5}) * mesh.nnodes))
c._call("CeedOperatorLinearAssemble{'PointBlock' if point_block else ''}Diagonal", op, d, None)
c._call("CeedVectorSetValue", w, ct.c_double(0.0))  # the output and the input have device arrays
c._call("CeedVectorScale", v, ct.c_double(1.0))
size = hip.fake_dev_bytes()
c._call("CeedMiOperatorApplyNoAlloc", op, v, w)
assert hip.fake_dev_bytes() == size
""")
