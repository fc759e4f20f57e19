"""The step clock and the wave speeds a step leaves for the next: every call that
changes the state, the time, the velocity or the kernel between steps, against
the oracle and against the same steps taken another way.  Two ways through the
same kernels agree bitwise; the oracle's steps to 1e-12 (as elsewhere)."""
import numpy as np
import pytest

import pyoracle as O
from helpers import noisy_state, rel_err, smooth_state
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu

# (physics, N, kernel): left wave speeds (packed columns, few batches;
# advection), and a kernel of their own in front of each step
PATHS = [("euler", 3, "mfma"), ("euler", 3, "simple"), ("euler", 4, "mfma_ws"), ("euler", 8, None),
         ("advection", 3, None)]


def _say(msg):
    print(f"[gpu-test] {msg}", flush=True)


def _solver(pb, physics, kernel, **kw):
    s = Solver(pb, physics, cfl=0.4, **kw)
    if kernel:
        s.set_stage_kernel(kernel)
    return s


@pytest.mark.parametrize("physics,N,kernel", PATHS)
def test_changes_between_steps(gpu, physics, N, kernel):
    """A new state, a new time and an rhs() between steps; step by step, in one
    call and replayed from graphs."""
    _say(f"clock {physics} N={N} {kernel}")
    pb = cube_problem(N, 2)
    ua, ub = noisy_state(pb, physics, seed=1), smooth_state(pb, physics, seed=2)
    o = O.Oracle(pb, physics, cfl=0.4)
    ra, da, _ = o.run(ua, 3)
    rb, db, _ = o.run(ub, 8)
    ends = []
    with _solver(pb, physics, kernel) as s:
        for way in ("steps", "call", "graph", "graph"):
            s.set_state(ua)
            s.set_time(1.5, 7)
            dts = s.step(3, return_dt=True)
            assert np.allclose(dts, da, rtol=1e-12, atol=0) and rel_err(s.get_state(), ra) < 1e-12
            t, dt, ts, done = s.time()
            assert ts == 10 and not done and dt == dts[2] and abs(t - 1.5 - dts.sum()) < 1e-14
            s.rhs(ua)  # (goes through the step's buffers)
            s.set_state(ub)
            if way == "steps":
                for i in range(8):
                    assert np.allclose(s.step(1, return_dt=True), db[i], rtol=1e-12, atol=0)
            elif way == "call":
                s.step(8, return_dt=True)
            else:
                s.step(8)
            ends.append((s.get_state(), s.time()))
            assert rel_err(ends[-1][0], rb) < 1e-12
    for u, tm in ends[1:]:
        assert np.array_equal(u, ends[0][0]) and tm == ends[0][1]


@pytest.mark.parametrize("physics,N,kernel", PATHS)
def test_past_tmax_and_back(gpu, physics, N, kernel):
    """Steps past tmax change nothing; a time set back makes them run again, on
    the state that is there."""
    pb = cube_problem(N, 2)
    u0 = noisy_state(pb, physics, seed=3)
    _, d, _ = O.Oracle(pb, physics, cfl=0.4).run(u0, 3)
    tmax = float(d[0] + d[1] + 0.5 * d[2])
    with _solver(pb, physics, kernel, tmax=tmax) as s:
        s.set_state(u0)
        dts = s.step(6, return_dt=True)
        t, _, ts, done = s.time()
        assert done and t == tmax and dts[2] < 0.6 * d[2] and not dts[3:].any()
        u = s.get_state()
        s.step(5)
        assert np.array_equal(u, s.get_state()) and s.time()[0] == tmax
        s.set_time(0.0, 0)
        dts = s.step(2, return_dt=True)
        ref, dref, _ = O.Oracle(pb, physics, cfl=0.4).run(u, 2)
        assert np.allclose(dts, dref, rtol=1e-12, atol=0) and rel_err(s.get_state(), ref) < 1e-12
        assert not s.time()[3]


def test_kernel_switched_between_steps(gpu):
    """Kernels that leave the wave speeds and kernels that do not, in turn."""
    pb = cube_problem(3, 3)
    u0 = noisy_state(pb, "euler", seed=4)
    ref, dref, _ = O.Oracle(pb, "euler", cfl=0.4).run(u0, 12)
    with Solver(pb, "euler", cfl=0.4) as s:
        s.set_state(u0)
        dts = []
        for k in ("mfma", "simple", "mfma_ws", "mfma", "mfma_ws", "simple"):
            s.set_stage_kernel(k)
            dts.append(s.step(2, return_dt=True))
        assert np.allclose(np.concatenate(dts), dref, rtol=1e-12, atol=0)
        assert rel_err(s.get_state(), ref) < 1e-12


def test_velocity_changed_between_steps(gpu):
    pb = cube_problem(3, 3)
    u0 = noisy_state(pb, "advection", seed=5)
    va, vb = (1.0, 0.3, -0.2), (-2.0, 1.0, 0.5)
    ra, da, _ = O.Oracle(pb, "advection", cfl=0.4, velocity=va).run(u0, 5)
    rb, db, _ = O.Oracle(pb, "advection", cfl=0.4, velocity=vb).run(ra, 5)
    for graphs in (False, True):
        with Solver(pb, "advection", cfl=0.4) as s:
            s.set_graphs(graphs)
            s.set_velocity(*va)
            s.set_state(u0)
            s.step(5)
            assert np.isclose(s.time()[1], da[-1], rtol=1e-12, atol=0)
            s.set_velocity(*vb)
            s.step(5)
            assert np.isclose(s.time()[1], db[-1], rtol=1e-12, atol=0)
            assert rel_err(s.get_state(), rb) < 1e-12


@pytest.mark.parametrize("n", [1, 1024, 1025, 1500])
def test_dt_histories(gpu, n):
    """Short histories come with the clock, longer ones by copy."""
    pb = cube_problem(1, 1)
    u0 = smooth_state(pb, "advection", seed=6)
    ref, dref, tref = O.Oracle(pb, "advection", cfl=0.4).run(u0, n)
    with Solver(pb, "advection", cfl=0.4) as s:
        s.set_state(u0)
        dts = s.step(n, return_dt=True)
        assert np.allclose(dts, dref, rtol=1e-12, atol=0) and s.time()[2] == n
        assert rel_err(s.get_state(), ref) < 1e-10  # rounding over n steps: n eps, with room


@pytest.mark.parametrize("physics,N", [("euler", 3), ("advection", 3)])
def test_recording_between_steps(gpu, physics, N):
    """Recorded steps and plain ones continue one another."""
    pb = cube_problem(N, 2)
    u0 = noisy_state(pb, physics, seed=7)
    ref, dref, tref = O.Oracle(pb, physics, cfl=0.4).run(u0, 9)
    with Solver(pb, physics, cfl=0.4) as s:
        s.set_state(u0)
        s.step(3)
        s.adjoint_record(3)
        dts = s.step(3, return_dt=True)
        assert np.allclose(dts, dref[6:], rtol=1e-12, atol=0)
        t, _, ts, _ = s.time()
        assert ts == 9 and abs(t - tref) < 1e-13 and rel_err(s.get_state(), ref) < 1e-12
