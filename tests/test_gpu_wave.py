"""The persistent one-wave-per-batch FP64 stage kernel: element counts that fill
no batch, several batches per wave, and more batches per wave than its table of
batch numbers holds at a time."""
import numpy as np
import pytest

import pyoracle as O
from helpers import noisy_state, rel_err_per_var
from test_gpu_cols import _check, _first_elements
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu-test] {msg}", flush=True)


@pytest.mark.parametrize("K", [1, 2, 4, 7, 25, 47])
@pytest.mark.parametrize("N", [3, 4])
def test_ragged_element_counts(gpu, N, K):
    _say(f"persistent ragged N={N} K={K}")
    full = cube_problem(N, 2)
    pb = _first_elements(full, K)
    u = np.ascontiguousarray(noisy_state(full, "euler", seed=N + K)[:, :K * full.Np])
    _check(pb, "euler", "lm", u, "mfma_ws")


@pytest.mark.parametrize("flux", ["lm", "rusanov"])
@pytest.mark.parametrize("N,nhex", [(3, 13), (4, 11)])
def test_several_batches_per_wave(gpu, N, nhex, flux):
    """More than one round, the last one partly filled and its last batch short
    (13,181 and 7985 elements)."""
    _say(f"persistent rounds N={N} {flux}")
    full = cube_problem(N, nhex)
    K = full.K - 1
    pb = _first_elements(full, K)
    u = np.ascontiguousarray(noisy_state(full, "euler", seed=N)[:, :K * full.Np])
    _check(pb, "euler", flux, u, "mfma_ws")


def test_many_batches_per_wave(gpu):
    """67 batches a wave (its numbers of batches come 64 at a time) against the
    packed-column kernel: the same sums of 168 terms in another order, 1e-12."""
    _say("persistent N=4 K=413,526")
    pb = cube_problem(4, 41)
    u = noisy_state(pb, "euler", seed=5)
    out = []
    for kernel in ("mfma", "mfma_ws"):
        with Solver(pb, "euler", cfl=0.4) as s:
            s.set_stage_kernel(kernel)
            s.set_state(u)
            s.step(1)
            out.append(s.get_state())
    assert max(rel_err_per_var(out[1], out[0])) < 1e-12
    assert np.abs(out[1] - out[0]).max() < 1e-11 * np.abs(out[0]).max()


def test_nan_stays_with_its_element(gpu):
    """A state that is not finite reaches its element and the neighbours that
    share a face with it, not the batch they are contracted in."""
    pb = cube_problem(4, 3)
    u = noisy_state(pb, "euler", seed=6)
    bad = 7
    u[2, bad * pb.Np + 3] = np.nan
    with Solver(pb, "euler", cfl=0.4) as s:
        out = []
        for kernel in ("mfma", "mfma_ws"):
            s.set_stage_kernel(kernel)
            r, _, _ = s.rhs(u)
            out.append(np.isnan(r.reshape(5, pb.K, pb.Np)).any(axis=(0, 2)))
    near = set((pb.arrays["vmapF"].reshape(pb.K, 4)[bad] // 4).tolist()) | {bad}
    for o in out:
        assert o[bad] and set(np.nonzero(o)[0].tolist()) <= near
