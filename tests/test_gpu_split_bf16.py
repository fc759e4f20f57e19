"""The split-BF16 stage kernel at order 4 on either side of the mesh size where its
fit is contracted in a rolled loop: as many 16-element batches as the GPU has
compute units, and one more."""
import numpy as np
import pytest
import torch

import pyoracle as O
from helpers import smooth_state
from test_gpu_cols import _first_elements
from test_gpu_parity import BF16, _term_scale
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("physics", ["euler", "advection"])
def test_rolled_and_whole_fit(gpu, physics, more):
    K = 16 * torch.cuda.get_device_properties(0).multi_processor_count + more
    print(f"[gpu-test] split-bf16 N=4 {physics} K={K}", flush=True)
    full = cube_problem(4, next(n for n in range(2, 40) if 6 * n ** 3 >= K))
    pb = _first_elements(full, K)
    u = np.ascontiguousarray(smooth_state(full, physics, seed=3)[:, :K * full.Np])
    with Solver(pb, physics, precision="bf16x6") as s:
        assert s.stage_kernel() == "mfma"
        r, _, _ = s.rhs(u)
    # (terms scale with |u| in advection, with |u|^2 in Euler)
    scale = _term_scale(pb, u) / (1.0 if physics == "euler" else np.abs(u).max())
    assert np.abs(r - O.Oracle(pb, physics).rhs(u)[0]).max() / scale < BF16["bf16x6"][0]
