"""Pass A of the Euler adjoint at order 1, where one wave takes eight elements:
element counts around a batch, and the exact trajectory gradient."""
import numpy as np
import pytest

from helpers import noisy_state
from test_gpu_adjoint_cols import _dot_product, dot
from test_gpu_cols import _first_elements
from traj_tl import Trajectory
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [2, 6, 8, 9, 15, 16, 41])
def test_adjoint_rhs_ragged(gpu, K):
    print(f"[gpu-test] adjoint rhs ragged euler N=1 K={K}", flush=True)
    full = cube_problem(1, 2)
    pb = _first_elements(full, K)
    _dot_product(pb, "euler", np.ascontiguousarray(noisy_state(full, "euler", seed=2)[:, :K * full.Np]), K)


@pytest.mark.parametrize("nhex", [3, 6])
def test_trajectory_gradient(gpu, nhex):
    """tau(u) and dt(u) included (162 elements: a short last batch; 1296: none), as at
    the other orders in test_gpu_adjoint_cols.py, same bound."""
    print(f"[gpu-test] trajectory gradient N=1 nhex={nhex}", flush=True)
    pb = cube_problem(1, nhex)
    u0 = noisy_state(pb, "euler", seed=3)
    rng = np.random.default_rng(5)
    wts = rng.uniform(0.5, 1.5, u0.shape)
    with Solver(pb, "euler", cfl=0.4) as s:
        s.set_state(u0)
        s.adjoint_record(6, 4)
        uT = s.get_state()
        grad = s.adjoint_backward(wts * uT)
        assert np.array_equal(s.adjoint_backward(wts * uT), grad)
    d = rng.standard_normal(u0.shape) * np.abs(u0)
    uTc, duT = Trajectory(pb, "euler", cfl=0.4).run(u0, 6, d)
    tl = dot(wts * uTc, duT)
    assert abs(dot(grad, d) - tl) <= 1e-10 * abs(tl)
