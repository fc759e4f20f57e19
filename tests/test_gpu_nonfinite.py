"""A state that is no longer a number is reported also where the run has an end time,
from both places that form wave speeds: the kernel in front of a step, and the last
stage of the step before."""
import numpy as np
import pytest

import pyoracle as O
from helpers import smooth_state
from exadglm_amd import _capi as A
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu

KERNELS = [(3, "mfma"), (3, "simple"), (4, "mfma"), (4, "mfma_ws"), (8, None)]


def _solver(pb, N, kernel):
    print(f"[gpu-test] not a number N={N} {kernel}", flush=True)
    s = Solver(pb, "euler", cfl=0.4, tmax=0.5)
    if kernel:
        s.set_stage_kernel(kernel)
    return s


def _reported(s):
    with pytest.raises(A.DGLMError) as ei:
        s.time()
    return ei.value.code == A.DGLM_ERR_STATE


@pytest.mark.parametrize("where", ["all", "one node"])
@pytest.mark.parametrize("N,kernel", KERNELS)
def test_state_given(gpu, N, kernel, where):
    """dt of the step is 0 and the clock says why; a sound state and a time set back
    run again."""
    pb = cube_problem(N, 3)
    good = smooth_state(pb, "euler", seed=8)
    bad = good.copy()
    if where == "all":
        bad[:] = np.nan
    else:
        bad[4, 5 * pb.Np + int(pb.arrays["Fmask"].ravel()[1])] = np.nan  # a face node of element 5
    with _solver(pb, N, kernel) as s:
        s.set_state(good)
        s.step(2)
        t = s.time()[0]
        s.set_state(bad)
        assert s.step(1, return_dt=True)[0] == 0.0
        assert _reported(s)
        s.step(3)
        assert _reported(s)
        s.set_state(good)
        s.set_time(t, 2)
        assert (s.step(3, return_dt=True) > 0).all() and s.time()[2] == 5


@pytest.mark.parametrize("N,kernel", [k for k in KERNELS if k[0] > 3])
def test_state_reached(gpu, N, kernel):
    """A NaN at a node inside an element is on its faces after a step: dt of the next
    one is 0."""
    pb = cube_problem(N, 3)
    u = smooth_state(pb, "euler", seed=9)
    inside = sorted(set(range(pb.Np)) - set(pb.arrays["Fmask"].ravel().tolist()))[0]
    dt = O.Oracle(pb, "euler", cfl=0.4).run(u, 1)[1][0]
    u[4, 5 * pb.Np + inside] = np.nan
    with _solver(pb, N, kernel) as s:
        s.set_state(u)
        dts = s.step(2, return_dt=True)
        assert abs(dts[0] - dt) < 1e-12 * dt and dts[1] == 0.0
        assert _reported(s)


def test_recorded_steps(gpu):
    pb = cube_problem(3, 3)
    u = smooth_state(pb, "euler", seed=10)
    u[0, 7 * pb.Np + int(pb.arrays["Fmask"].ravel()[0])] = np.nan
    with _solver(pb, 3, None) as s:
        s.set_state(u)
        s.adjoint_record(2)
        assert _reported(s)


def test_velocity_given(gpu):
    pb = cube_problem(2, 3)
    v = np.ones((3, pb.K * pb.Np))
    v[0, 7 * pb.Np + int(pb.arrays["Fmask"].ravel()[0])] = np.nan
    with Solver(pb, "advection", cfl=0.4, tmax=0.5) as s:
        s.set_velocity(*v)
        s.set_state(smooth_state(pb, "advection", seed=1))
        s.step(2)
        assert _reported(s)
