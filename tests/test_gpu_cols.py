"""The packed-column FP64 stage kernel: both of its configurations (few and many
elements per workgroup), ragged element counts, both fluxes, against the oracle."""
import types

import numpy as np
import pytest

import pyoracle as O
from helpers import noisy_state, rel_err_per_var
from exadglm_amd.problem import cube_problem
from exadglm_amd.solver import Solver

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu-test] {msg}", flush=True)


def _first_elements(pb, K):
    """The first K elements of a mesh as a mesh of their own: faces whose
    neighbour is cut off become boundary faces (u+ = u-), tagged 0."""
    a = {k: v.copy() for k, v in pb.arrays.items()}
    Np, Nfp = pb.Np, pb.Nfp
    for n in ("Fscale", "nx", "ny", "nz", "EtoB", "px", "py", "pz", "rx", "ry", "rz", "sx", "sy", "sz", "tx", "ty",
              "tz"):
        a[n] = np.ascontiguousarray(a[n][:K])
    Fm = a["Fmask"].reshape(4, Nfp)
    vM = (np.arange(K)[:, None, None] * Np + Fm[None]).astype(np.int32)
    vP = a["vmapP"].reshape(pb.K, 4, Nfp)[:K]
    cut = a["vmapF"].reshape(pb.K, 4)[:K] >= 4 * K
    own = np.arange(4 * K, dtype=np.int32).reshape(K, 4)
    a["vmapF"] = np.ascontiguousarray(np.where(cut, own, a["vmapF"].reshape(pb.K, 4)[:K]).astype(np.int32))
    a["vmapP"] = np.ascontiguousarray(np.where(cut[:, :, None], vM, vP).astype(np.int32))
    a["EtoB"] = np.zeros((K, 4), np.int32)
    return types.SimpleNamespace(N=pb.N, K=K, Np=Np, Nfp=Nfp, arrays=a)


def _check(pb, physics, flux, u, kernel, steps=2):
    vel = (1.0, -0.4, 0.7)
    o = O.Oracle(pb, physics, cfl=0.4, flux=flux, velocity=vel if physics == "advection" else None)
    with Solver(pb, physics, cfl=0.4, flux=flux) as s:
        if kernel is not None:
            s.set_stage_kernel(kernel)
        if physics == "advection":
            s.set_velocity(*vel)
        r, _, _ = s.rhs(u)
        s.set_state(u)
        s.step(steps)
        un = s.get_state()
    assert max(rel_err_per_var(r, o.rhs(u)[0])) < 1e-12
    assert max(rel_err_per_var(un, o.run(u, steps)[0])) < 1e-12


@pytest.mark.parametrize("flux", ["lm", "rusanov"])
@pytest.mark.parametrize("physics,N,nhex", [("euler", 1, 13), ("euler", 2, 11), ("euler", 3, 11), ("euler", 4, 17),
                                            ("euler", 5, 11), ("euler", 6, 13), ("euler", 7, 5), ("euler", 10, 3), ("euler", 3, 15),
                                            ("euler", 5, 15),
                                            ("advection", 1, 13), ("advection", 2, 13), ("advection", 5, 18),
                                            ("advection", 6, 18), ("advection", 8, 5)])
def test_large_meshes(gpu, physics, N, nhex, flux):
    """Meshes just past the size where the large configuration of the order
    starts (orders with one configuration: several workgroups), the last batch
    short where its size does not divide 6 nhex^3."""
    _say(f"packed columns {physics} N={N} K={6 * nhex ** 3} {flux}")
    pb = cube_problem(N, nhex)
    _check(pb, physics, flux, noisy_state(pb, physics, seed=N), "mfma" if N <= 6 else None)


@pytest.mark.parametrize("K", [1, 2, 17, 25])
@pytest.mark.parametrize("physics", ["euler", "advection"])
@pytest.mark.parametrize("N", range(1, 11))
def test_ragged_element_counts(gpu, physics, N, K):
    """Element counts that fill no batch, down to a single element; K*Np odd at
    N = 4 and 8 (rows at 8-byte alignment)."""
    _say(f"packed columns ragged {physics} N={N} K={K}")
    full = cube_problem(N, 2)
    pb = _first_elements(full, K)
    u = np.ascontiguousarray(noisy_state(full, physics, seed=N + K)[:, :K * full.Np])
    _check(pb, physics, "lm", u, "mfma" if N <= 6 else None)


@pytest.mark.parametrize("N,nhex,kernel", [(3, 3, "mfma"), (3, 13, "mfma"), (3, 16, "mfma_ws"), (4, 11, "mfma"),
                                           (4, 16, "mfma_ws"), (5, 3, "mfma"), (8, 2, "simple")])
def test_kernel_chosen(gpu, N, nhex, kernel):
    """FP64 Euler: the persistent kernel only at N = 3, 4 on meshes that fill its
    waves (2048, with 6 and 3 elements a round)."""
    with Solver(cube_problem(N, nhex), "euler") as s:
        assert s.stage_kernel() == kernel
