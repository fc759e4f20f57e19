"""Dirichlet faces on meshes that the FP64 kernels go through in several rounds: the
persistent kernel with more batches than waves (and more than its table of batch
numbers holds), the packed-column kernel in its large configurations, the last batch
short; against the oracle, with the prescribed states changed between the steps."""
import numpy as np
import pytest

import pyoracle as O
from helpers import noisy_state, rel_err_per_var
from test_gpu_cols import _first_elements
from test_gpu_features import _relabel
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu
CUT = {"x": "bc1", "y": "pbc", "z": "bc1"}
WAVES, EB = 2048, {3: 6, 4: 3}  # of the persistent kernel on 256 compute units; its elements a batch


def _say(msg):
    print(f"[gpu-test] {msg}", flush=True)


def _open_box(N, nhex, drop):
    """The box without its last elements; the faces on its open sides stay Dirichlet
    faces, those of the cut take u+ = u-."""
    full = cube_problem(N, nhex, bc=CUT)
    pb = _first_elements(full, full.K - drop)
    pb.arrays["EtoB"] = np.ascontiguousarray(full.arrays["EtoB"].reshape(full.K, 4)[:pb.K])
    return full, pb


def _states(pb, u, seed):
    """A prescribed state on every face node: the interior trace with 5% noise."""
    at = np.arange(pb.K)[:, None] * pb.Np + pb.arrays["Fmask"].reshape(1, -1)
    g = u[:, at.ravel()]
    return g * (1 + 0.05 * np.random.default_rng(seed).standard_normal(g.shape))


def _check(pb, physics, flux, kernel, u):
    gs = [_states(pb, u, seed) for seed in (1, 2)]
    o = O.Oracle(pb, physics, cfl=0.4, flux=flux)
    with Solver(pb, physics, cfl=0.4, flux=flux) as s:
        s.set_stage_kernel(kernel)
        assert s.stage_kernel() == kernel and len(s.dirichlet_faces())
        s.set_dirichlet(gs[0])
        o.set_dirichlet(gs[0])
        assert max(rel_err_per_var(s.rhs(u)[0], o.rhs(u)[0])) < 1e-12
        s.set_state(u)
        ref = u
        for g in gs:
            s.set_dirichlet(g)
            o.set_dirichlet(g)
            s.step(1)
            ref = o.run(ref, 1)[0]
        assert max(rel_err_per_var(s.get_state(), ref)) < 1e-12


@pytest.mark.parametrize("flux", ["lm", "rusanov"])
@pytest.mark.parametrize("N,nhex", [(3, 13), (4, 11)])
def test_persistent_kernel(gpu, N, nhex, flux):
    _say(f"open box persistent N={N} {flux}")
    full, pb = _open_box(N, nhex, 1)
    assert -(-pb.K // EB[N]) > WAVES and pb.K % EB[N]
    _check(pb, "euler", flux, "mfma_ws", np.ascontiguousarray(noisy_state(full, "euler", seed=N)[:, :pb.K * pb.Np]))


@pytest.mark.parametrize("flux", ["lm", "rusanov"])
@pytest.mark.parametrize("physics,N,nhex", [("euler", 1, 13), ("euler", 2, 11), ("euler", 3, 15), ("euler", 4, 15),
                                            ("euler", 5, 15), ("euler", 6, 13), ("advection", 3, 12),
                                            ("advection", 5, 12)])
def test_packed_columns(gpu, physics, N, nhex, flux):
    _say(f"open box packed columns {physics} N={N} {flux}")
    full, pb = _open_box(N, nhex, 1)
    _check(pb, physics, flux, "mfma", np.ascontiguousarray(noisy_state(full, physics, seed=N)[:, :pb.K * pb.Np]))


def test_many_batches_per_wave(gpu):
    """67 batches a wave, against the packed-column kernel: the same sums of 168 terms
    in another order, 1e-12."""
    _say("open box persistent N=4 K=413,525")
    full, pb = _open_box(4, 41, 1)
    assert -(-pb.K // EB[4]) > 64 * WAVES and pb.K % EB[4]
    u = np.ascontiguousarray(noisy_state(full, "euler", seed=5)[:, :pb.K * pb.Np])
    g = _states(pb, u, 3)
    out = []
    for kernel in ("mfma", "mfma_ws"):
        with Solver(pb, "euler", cfl=0.4) as s:
            s.set_stage_kernel(kernel)
            s.set_dirichlet(g)
            s.set_state(u)
            s.step(1)
            out.append(s.get_state())
    assert max(rel_err_per_var(out[1], out[0])) < 1e-12


@pytest.mark.parametrize("N,nhex", [(3, 13), (4, 11)])
def test_order_of_the_elements(gpu, N, nhex):
    """The persistent kernel's visiting order is a schedule only, also with several
    batches a wave and a short last one: a relabelled mesh and one without node
    coordinates give the same bits."""
    _say(f"persistent element order N={N}")
    full = cube_problem(N, nhex)
    pb = _first_elements(full, full.K - 1)
    K, Np = pb.K, pb.Np
    assert -(-K // EB[N]) > WAVES and K % EB[N]
    u0 = np.ascontiguousarray(noisy_state(full, "euler", seed=6)[:, :K * Np])
    arr, old = _relabel(pb, 12)
    no_xyz = {k: v for k, v in pb.arrays.items() if k not in ("px", "py", "pz")}
    runs = []
    for arrays, u in ((pb.arrays, u0), (arr, np.ascontiguousarray(u0.reshape(5, K, Np)[:, old].reshape(5, -1))),
                      (no_xyz, u0)):
        with Solver(pb, "euler", cfl=0.4, arrays=arrays, K=K, flux="rusanov") as s:
            s.set_stage_kernel("mfma_ws")
            s.set_state(u)
            s.step(2)
            runs.append(s.get_state())
    back = np.empty((5, K, Np))
    back[:, old] = runs[1].reshape(5, K, Np)
    assert np.isfinite(runs[0]).all()
    assert np.array_equal(runs[0], back.reshape(5, -1)) and np.array_equal(runs[0], runs[2])
