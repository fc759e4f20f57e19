"""dt of a mesh with elements of negative volume (their Fscale is negative): the
largest lambda * Fscale of the others."""
import types

import numpy as np
import pytest

import pyoracle as O
from helpers import smooth_state
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("physics,kernel", [("euler", "mfma"), ("euler", "mfma_ws"), ("advection", None)])
def test_dt_passes_over_negative_fscale(gpu, physics, kernel):
    """The first 1024 elements of 1296 inside out: sixteen workgroups of the wave-speed
    kernel (64 elements), one for each part of the maximum, hold nothing positive."""
    print(f"[gpu-test] inside-out elements {physics} {kernel}", flush=True)
    full = cube_problem(3, 6)
    a = {k: v.copy() for k, v in full.arrays.items()}
    a["Fscale"].reshape(full.K, 4)[:1024] *= -1
    pb = types.SimpleNamespace(N=full.N, K=full.K, Np=full.Np, Nfp=full.Nfp, arrays=a)
    u = smooth_state(full, physics, seed=4)
    dt = O.Oracle(pb, physics, cfl=0.4).run(u, 1)[1][0]
    with Solver(pb, physics, cfl=0.4) as s:
        if kernel:
            s.set_stage_kernel(kernel)
        s.set_state(u)
        got = s.step(1, return_dt=True)[0]
    assert dt > 0 and abs(got - dt) < 1e-14 * dt
