"""Pass A of the adjoint on packed columns: the orders and element counts the
dot-product tests of test_gpu_adjoint.py leave out, and the exact trajectory
gradient at orders above 3."""
import numpy as np
import pytest

import pyoracle as O
from helpers import noisy_state
from test_gpu_cols import _first_elements
from traj_tl import Trajectory
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu-test] {msg}", flush=True)


def dot(a, b):
    return float(np.dot(np.ravel(a), np.ravel(b)))


def _dot_product(pb, physics, u, seed):
    """<J du, rbar> (oracle tangent-linear, tau frozen) = <du, J^T rbar>, to the
    rounding of sums of this length (1e-13 of the norms)."""
    rng = np.random.default_rng(seed)
    du = rng.standard_normal(u.shape)
    rbar = rng.standard_normal(u.shape)
    with Solver(pb, physics) as s:
        ubar, taubar = s.adjoint_rhs(u, rbar)
    o = O.Oracle(pb, physics)
    tl = O.rhs_tl(o, u, du)
    lhs, rhs = dot(tl, rbar), dot(du, ubar)
    assert abs(lhs - rhs) <= 1e-13 * np.linalg.norm(tl) * np.linalg.norm(rbar), (lhs, rhs)
    # taubar: the RHS is affine in tau, so its difference is exact up to rounding
    dtau = rng.standard_normal((pb.K, 4))
    _, _, tau = o.rhs(u)
    d = O.rhs_tau(o, u, tau + dtau) - O.rhs_tau(o, u, tau)
    lhs, rhs = dot(d, rbar), dot(taubar, dtau)
    assert abs(lhs - rhs) <= 1e-11 * np.linalg.norm(d) * np.linalg.norm(rbar), (lhs, rhs)


@pytest.mark.parametrize("physics", ["advection", "euler"])
@pytest.mark.parametrize("N", range(1, 11))
def test_adjoint_rhs_every_order(gpu, physics, N):
    _say(f"adjoint rhs {physics} N={N}")
    pb = cube_problem(N, 3 if N <= 6 else 2)
    _dot_product(pb, physics, noisy_state(pb, physics, seed=N + 51), N)


@pytest.mark.parametrize("K", [1, 7, 17])
@pytest.mark.parametrize("physics", ["advection", "euler"])
@pytest.mark.parametrize("N", [1, 4, 5, 8, 9, 10])
def test_adjoint_rhs_ragged(gpu, physics, N, K):
    """Element counts that fill no workgroup, boundary faces (u+ = u-)."""
    _say(f"adjoint rhs ragged {physics} N={N} K={K}")
    full = cube_problem(N, 2)
    pb = _first_elements(full, K)
    _dot_product(pb, physics, np.ascontiguousarray(noisy_state(full, physics, seed=N)[:, :K * full.Np]), N + K)


@pytest.mark.parametrize("N", [2, 4, 5, 7])
def test_euler_trajectory_gradient(gpu, N):
    """J = 1/2 sum w u(T)^2 after 6 steps, tau(u) and dt(u) included: the gradient
    along random directions equals the CPU tangent-linear of the oracle
    trajectory to rounding (as at N = 3 in test_gpu_adjoint.py)."""
    _say(f"trajectory gradient N={N}")
    pb = cube_problem(N, 3 if N <= 5 else 2)
    u0 = noisy_state(pb, "euler", seed=3)
    rng = np.random.default_rng(5)
    wts = rng.uniform(0.5, 1.5, u0.shape)
    T = Trajectory(pb, "euler", cfl=0.4)
    with Solver(pb, "euler", cfl=0.4) as s:
        s.set_state(u0)
        s.adjoint_record(6, 4)
        uT = s.get_state()
        grad = s.adjoint_backward(wts * uT)
    for _ in range(2):
        d = rng.standard_normal(u0.shape) * np.abs(u0)
        uTc, duT = T.run(u0, 6, d)
        tl = dot(wts * uTc, duT)
        assert abs(dot(grad, d) - tl) <= 1e-10 * abs(tl)


def test_advection_recording_keeps_no_states(gpu):
    """Advection is linear: the reverse sweep needs no states, so the tape does not
    grow with the checkpoint interval or the kept segments, a repeated sweep gives
    the same gradient, and <S du, w> = <du, S^T w> holds over a second recording
    of another length."""
    _say("advection recording")
    pb = cube_problem(5, 3)
    rng = np.random.default_rng(3)
    du, w = rng.standard_normal((2, 1, pb.K * pb.Np))
    with Solver(pb, "advection", cfl=0.5) as s:
        s.set_velocity(1.0, 0.5, -0.25)
        res = []
        for n, every, keep in ((9, 4, -1), (9, 2, 0), (12, 5, 1)):
            s.set_adjoint_keep(keep)
            s.set_state(du)
            s.set_time(0.0, 0)
            s.adjoint_record(n, every)
            Sdu = s.get_state()
            g = s.adjoint_backward(w)
            np.testing.assert_array_equal(s.adjoint_backward(w), g)
            lhs, rhs = dot(Sdu, w), dot(du, g)
            assert abs(lhs - rhs) <= 1e-12 * np.linalg.norm(Sdu) * np.linalg.norm(w)
            res.append((g, s.tape_bytes()))
    np.testing.assert_array_equal(res[0][0], res[1][0])
    assert res[0][1] == res[1][1]
