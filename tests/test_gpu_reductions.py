"""The reductions of the time integrator's vector kernels against sums on the host, through the launch functions themselves: a
solver converges with wrong sums too, so its solution says nothing about them.  Lengths below a block of 512, at its edges, with a
ragged last block, and past one and two passes of the largest grid (256 blocks); every count of vectors in a row of 8 and
several rows.  The inputs are small integers, whose products and sums are exact in FP64: a missing or doubled entry shows."""
import ctypes as ct
import sys

import numpy as np
import pytest

from pyhonee import ts as TS

pytestmark = pytest.mark.gpu

SLOTS, BLOCKS, MAX_LINCOMB = 32, 256, 8
PASS = BLOCKS * 512
LENGTHS = [1, 511, 512, 513, PASS - 1, PASS + 1, 2 * PASS + 777]
EPS = np.finfo(np.float64).eps


class Publish(ct.Structure):
    _fields_ = [("h", ct.c_void_p), ("flag", ct.c_void_p), ("seq", ct.c_ulonglong), ("count", ct.c_int)]


class LinComb(ct.Structure):
    _fields_ = [("m", ct.c_int), ("c", ct.c_double * MAX_LINCOMB), ("x", ct.c_void_p * MAX_LINCOMB)]


class RkStage(ct.Structure):
    _fields_ = [("d", ct.c_void_p), ("r", ct.c_void_p), ("q", ct.c_void_p), ("k", ct.c_void_p), ("y", ct.c_void_p), ("ck", ct.c_double),
                ("lc", LinComb)]


# C++ names of the launch functions (krylov.hpp)
MDOT = "_Z11launch_mdotPKdS0_xixPdP12ihipStream_t"
DOT = "_Z10launch_dotPKdS0_xiPdS1_P12ihipStream_tRK7Publish"
PROJECT = "_Z18launch_project_outPdPKdxixiS_S_P12ihipStream_t"
NORMALIZE = "_Z16launch_normalizePdPKdiS_xP12ihipStream_tRK7Publish"
COUNT = "_Z22launch_count_nonfinitePKdxiPdS1_P12ihipStream_tRK7Publish"
RK_LAST = "_Z14launch_rk_lastRK7RkStagexiPdS2_P12ihipStream_tRK7Publish"
PB_INVERT = "_Z16launch_pb_invertPdxiS_S_P12ihipStream_tRK7Publish"


class Launcher:
    def __init__(self):
        import torch

        self.torch, self.lib = torch, TS.load_ts_lib()
        self.partial = torch.full((SLOTS, BLOCKS), np.nan, dtype=torch.float64, device="cuda:0")
        self.out = torch.full((SLOTS,), np.nan, dtype=torch.float64, device="cuda:0")

    def put(self, a):
        return self.torch.tensor(np.ascontiguousarray(a), device="cuda:0")

    def __call__(self, name, *args):
        conv = {self.torch.Tensor: lambda t: ct.c_void_p(t.data_ptr()), int: ct.c_longlong}
        args = [a if isinstance(a, (ct._SimpleCData, ct.Structure)) or a is None else conv[type(a)](a) for a in args]
        args = [ct.byref(a) if isinstance(a, ct.Structure) else a for a in args]
        assert getattr(self.lib, name)(*args) == 0, name

    def result(self, slot):
        self.torch.cuda.synchronize()
        return float(self.out[slot])


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n", LENGTHS)
def test_arnoldi_step(n):
    L, rng = Launcher(), np.random.default_rng(n)
    for k in (1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17, 31):
        _say(f"reductions arnoldi n={n} k={k}")
        w, V = rng.integers(-8, 9, n).astype(float), rng.integers(-3, 4, (k, n)).astype(float)
        V[:, -1], w[-1] = 3, 8
        h = V @ w
        dw, dV = L.put(w), L.put(V)
        L.partial.fill_(np.nan)
        L(MDOT, dw, dV, n, ct.c_int(k), n, L.partial, None)
        L(PROJECT, dw, dV, n, ct.c_int(k), n, ct.c_int(k), L.partial, L.out, None)
        L.torch.cuda.synchronize()
        assert (L.out[:k].cpu().numpy() == h).all(), k
        w -= h @ V
        assert (dw.cpu().numpy() == w).all(), k
        L(NORMALIZE, dw, L.partial, ct.c_int(k), L.out, n, None, Publish())
        # a sum of n positive terms in blocks: (terms a thread + tree) roundings, under 64 here
        ss = float(w @ w)
        assert abs(L.result(k) - ss) <= 64 * EPS * ss
        if ss > 0:
            assert np.allclose(dw.cpu().numpy(), w / np.sqrt(ss), rtol=64 * EPS, atol=0)


@pytest.mark.parametrize("n", LENGTHS)
def test_dot_and_nonfinite_count(n):
    _say(f"reductions dot n={n}")
    L, rng = Launcher(), np.random.default_rng(n)
    x, y = rng.integers(1, 9, n).astype(float), rng.integers(1, 9, n).astype(float)
    dx, dy = L.put(x), L.put(y)
    L(DOT, dx, dy, n, ct.c_int(3), L.partial, L.out, None, Publish())
    assert L.result(3) == x @ y
    one = L.put(np.ones(n))
    for at in {0, n - 1, n // 2, (n - 1) // 512 * 512, min(n - 1, PASS - 1), min(n - 1, PASS)}:
        for bad in (np.nan, np.inf, -np.inf):
            z = x.copy()
            z[at] = bad
            dz = L.put(z)
            L(COUNT, dz, n, ct.c_int(0), L.partial, L.out, None, Publish())
            assert L.result(0) == 1, (at, bad)
            # the last Runge-Kutta stage: y = q + 2 d r, with the bad entry in q
            res = L.put(np.zeros(n))
            a = RkStage(d=one.data_ptr(), r=dy.data_ptr(), q=dz.data_ptr(), k=None, y=res.data_ptr(), ck=2.0)
            L(RK_LAST, a, n, ct.c_int(1), L.partial, L.out, None, Publish())
            assert L.result(1) == 1, (at, bad)
            assert np.array_equal(res.cpu().numpy(), z + 2 * y, equal_nan=True)


@pytest.mark.parametrize("nodes", [1, 255, 257, BLOCKS * 256 - 1, BLOCKS * 256 + 300])
def test_block_inverse(nodes):
    _say(f"reductions pb_invert nodes={nodes}")
    L, rng = Launcher(), np.random.default_rng(nodes)
    A = rng.uniform(-1, 1, (nodes, 5, 5)) + 6 * np.eye(5)  # diagonally dominant: condition below 20
    ref = np.linalg.inv(A)
    dA = L.put(A)
    L(PB_INVERT, dA, nodes, ct.c_int(0), L.partial, L.out, None, Publish())
    assert L.result(0) == 0
    assert np.abs(dA.cpu().numpy() - ref).max() < 100 * EPS * np.abs(ref).max()
    for at in {0, nodes - 1, min(nodes - 1, BLOCKS * 256)}:
        B = A.copy()
        B[at, :, 2] = 0
        L(PB_INVERT, L.put(B), nodes, ct.c_int(0), L.partial, L.out, None, Publish())
        assert L.result(0) == 1, at


@pytest.mark.parametrize("gmres", [0, 1])
def test_step_fails_on_nonfinite_state(gmres):
    """The counts as the integrator reads them: a state with one bad entry ends the step with an error."""
    from pyhonee import mesh as M
    from pyhonee import problems as PR
    from pyhonee.driver import NewtonianProblem, context_from_dict

    mesh, tab = M.box_mesh((3, 3, 3), 1, lengths=(1.0, 1.0, 1.0)), M.tabulate(1, 0)
    d = PR.tgv_context_dict(state_var=0, stabilization=0, implicit=False, dt=1e-3, tau=PR.default_tau(1))
    q0 = PR.q_from_prim(PR.TGV_GAS, PR.nodal_field(mesh, lambda x: PR.taylor_green_prim(x)), 0).ravel()
    prob = NewtonianProblem(mesh, tab, context_from_dict(d), 0)
    ts = TS.TimeStepper(prob, TS.default_options(type=TS.TS_RK, rk_type=TS.RK_EULER, dt=1e-3, mass_gmres=gmres, mass_max_it=3))
    for at in (0, len(q0) // 2, len(q0) - 1):
        for bad in (np.nan, np.inf):
            _say(f"reductions step gmres={gmres} at={at} bad={bad}")
            q = q0.copy()
            q[at] = bad
            ts.set_solution(q, 0.0)
            with pytest.raises(RuntimeError, match="non-finite"):
                ts.step(1)
    ts.set_solution(q0, 0.0)
    ts.step(1)
    ts.close()
    prob.close()
