"""The work that the solver is measured on: what a program does with a context
once its mesh and initial state are in hand.

A pass sets the state and the time, advances a number of LSRK4(5) steps (or
records them and sweeps back) and takes the result, all through the Python
binding of the C ABI.  The meshes are uniform boxes of (nx, ny, nz) hexes x 6
tetrahedra.  Kinds of pass:

  steps      step(n) with nothing coming back per step (graph replay)
  chunk      step(n, return_dt=True) and time(): one output interval of the launcher
  dirichlet  n times: new boundary states on the open faces, then one step
  adjoint    dglm_evolve and its backward (checkpointed recording, reverse sweep)

States are what such runs hold in earnest: the isentropic vortex (Euler) or a
random Fourier field (advection) with a smooth random perturbation and small
jumps between elements, as every computed discontinuous Galerkin state has.
"""
import functools
import math

import numpy as np
import torch

from exadglm_amd.autograd import dglm_evolve
from exadglm_amd.problem import uniform_problem
from exadglm_amd.solver import Solver

GAMMA = 1.4
TAU_SCALE = 1.2
VELOCITY = (1.0, 0.5, 0.25)
RKA = (0.0, -567301805773.0 / 1357537059087.0, -2404267990393.0 / 2016746695238.0,
       -3550918686646.0 / 2091501179385.0, -1275806237668.0 / 842570457699.0)
RKB = (1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0,
       1720146321549.0 / 2090206949498.0, 3134564353537.0 / 4481467310338.0,
       2277821191437.0 / 14882151754819.0)


def _case(name, kind, physics, N, nx, ny, nz, steps, flux="lm", precision="fp64", cfl=0.4, every=0, keep=-1):
    c = dict(kind=kind, physics=physics, N=N, nx=nx, ny=ny, nz=nz, steps=steps, flux=flux, precision=precision,
             cfl=cfl)
    if kind == "adjoint":
        c.update(every=every, keep=keep)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one step of a tiny mesh, dt and time read back (a coupled step loop)
        _case("euler_n4_k384_one_step", "chunk", "euler", 4, 4, 4, 4, 1),
        # the small advection configuration: K = 6000, upwind flux
        _case("advection_n3_k6000", "steps", "advection", 3, 10, 10, 10, 10, flux="rusanov", cfl=0.5),
        # one output interval of the advection notebook run (6^3 hexes, N = 5, 809 steps, 30 outputs)
        _case("advection_n5_k1296_chunk", "chunk", "advection", 5, 6, 6, 6, 20, cfl=0.8),
        # one output interval of the Euler notebook run (6^3 hexes, N = 5, 1318 steps, 30 outputs)
        _case("euler_n5_k1296_chunk", "chunk", "euler", 5, 6, 6, 6, 40, cfl=0.8),
        # an ordinary run on a box whose sides and element count fit no tile
        _case("euler_n3_k44574", "steps", "euler", 3, 23, 19, 17, 4),
        # the headline run: the vortex at N = 4, K = 196,608, Rusanov flux
        _case("euler_n4_k196608", "steps", "euler", 4, 32, 32, 32, 4, flux="rusanov"),
        # the N = 6 vortex, K = 82,944, in FP64 and with the FP32 contraction
        _case("euler_n6_k82944", "steps", "euler", 6, 24, 24, 24, 3, flux="rusanov"),
        _case("euler_n6_k82944_fp32", "steps", "euler", 6, 24, 24, 24, 3, flux="rusanov", precision="fp32"),
        # high order: what the orders above 6 are for, few elements with many nodes
        _case("euler_n8_k6000", "steps", "euler", 8, 10, 10, 10, 3),
        # open box in x and z, boundary states replaced before every step
        _case("euler_n4_k11520_dirichlet", "dirichlet", "euler", 4, 16, 12, 10, 4),
        # the Euler adjoint at full size: of two checkpoint segments one kept whole, one recomputed
        _case("adjoint_euler_n4_k196608", "adjoint", "euler", 4, 32, 32, 32, 6, every=3, keep=1),
        # the advection adjoint configuration: N = 5, K = 48,000, every segment kept (the default)
        _case("adjoint_advection_n5_k48000", "adjoint", "advection", 5, 20, 20, 20, 20, cfl=0.5, every=5),
    ]


def draw(rng):
    kind = rng.choices(("steps", "chunk", "dirichlet", "adjoint"), (5, 3, 1.5, 2.5))[0]
    physics = rng.choices(("euler", "advection"), (7, 3))[0]
    top = 6 if kind == "adjoint" else 10
    N = rng.choices(range(1, top + 1), (1, 2, 4, 5, 4, 4, 1, 1, 0.5, 0.5)[:top])[0]
    Np = (N + 1) * (N + 2) * (N + 3) // 6
    # nodes of the mesh; the high orders and the long chunks stay smaller
    most = 3e6 if N <= 6 else 6e5
    most = 4e5 if kind == "chunk" else most
    hexes = 10 ** rng.uniform(math.log10(5e3), math.log10(most)) / Np / 6
    side = [max(3, round(hexes ** (1 / 3) * rng.uniform(0.75, 1.3))) for _ in range(3)]
    precision = "fp64"
    if kind in ("steps", "chunk") and N <= 6:
        precision = rng.choices(("fp64", "fp32", "bf16x6"), (6, 3, 1))[0]
    steps = rng.randint(3, 6) if kind != "chunk" else rng.randint(5, 30)
    flux = "lm" if kind == "adjoint" else rng.choice(("lm", "rusanov"))
    cfl = rng.choice((0.4, 0.5, 0.8)) if flux == "lm" else rng.choice((0.4, 0.5))
    return _case(None, kind, physics, N, *side, steps, flux=flux, precision=precision, cfl=cfl,
                 every=rng.randint(2, 3), keep=rng.choice((-1, -1, 0, 1)))


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


@functools.lru_cache(maxsize=2)
def _problem(N, nx, ny, nz, is_open):
    bc = {"x": "bc1", "y": "pbc", "z": "bc1"} if is_open else None
    return uniform_problem(N, nx + 1, ny + 1, nz + 1, box=(0.0, 10.0, 0.0, 10.0, 0.0, 10.0 / 3.0), bc=bc)


def _problem_of(case):
    return _problem(case["N"], case["nx"], case["ny"], case["nz"], case["kind"] == "dirichlet")


def _points(pb):
    return [torch.as_tensor(np.array(pb.arrays[c]), device=_device()).reshape(-1) for c in ("px", "py", "pz")]


def _waves(rng, x, y, z, n=4):
    """Random Fourier field of the box, amplitude about one."""
    out = torch.zeros_like(x)
    for _ in range(n):
        k = rng.integers(-2, 3, 3)
        amp, phase = rng.uniform(0.3, 1.0) / n, rng.uniform(0, 2 * math.pi)
        out += amp * torch.cos((2 * math.pi / 10) * (float(k[0]) * x + float(k[1]) * y + 3 * float(k[2]) * z) + phase)
    return out


def _state(case, x, y, z, seed, t=0.0):
    """Conserved variables at the points: a field of the seed, displaced by t."""
    rng = np.random.default_rng(seed)
    if case["physics"] == "advection":
        return _waves(rng, x - VELOCITY[0] * t, y - VELOCITY[1] * t, z - VELOCITY[2] * t, 8)[None].clone()
    xc, yc = rng.uniform(3, 7, 2) + t
    du, dv, dT = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x)
    beta = 5.0
    for ix in (-1, 0, 1):
        for iy in (-1, 0, 1):
            dx, dy = x - (xc % 10 + 10 * ix), y - (yc % 10 + 10 * iy)
            ex = torch.exp(0.5 * (1 - dx * dx - dy * dy))
            du -= beta / (2 * math.pi) * dy * ex
            dv += beta / (2 * math.pi) * dx * ex
            dT -= (GAMMA - 1) * beta * beta / (8 * GAMMA * math.pi ** 2) * ex * ex
    rho = (1 + dT) ** (1 / (GAMMA - 1))
    p = rho ** GAMMA
    rho = rho * (1 + 0.01 * _waves(rng, x, y, z))
    p = p * (1 + 0.01 * _waves(rng, x, y, z))
    u, v, w = 1 + du, 1 + dv, 0.1 * _waves(rng, x, y, z)
    return torch.stack([rho, rho * u, rho * v, rho * w, p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v + w * w)])


def _initial(case, pb, seed):
    u = _state(case, *_points(pb), seed)
    g = torch.Generator().manual_seed(seed)
    jump = torch.randn(u.shape[0], pb.K, 1, generator=g, dtype=torch.float64).to(u.device)
    return (u.view(u.shape[0], pb.K, pb.Np) * (1 + 1e-6 * jump)).reshape(u.shape).contiguous()


def _open_faces(pb):
    return np.flatnonzero(pb.arrays["EtoB"].reshape(-1) == 1)


def _boundary(case, pb, seed):
    """The boundary states of each step, [steps][nvar][nd][Nfp]."""
    faces = _open_faces(pb)
    nodes = ((faces // 4)[:, None] * pb.Np + pb.arrays["Fmask"].reshape(4, -1)[faces % 4]).ravel()
    at = [q[torch.as_tensor(nodes, device=q.device)] for q in _points(pb)]
    return [_state(case, *at, seed, t=1e-3 * i).reshape(-1, len(faces), pb.Nfp).contiguous()
            for i in range(case["steps"])]


def _cotangent(case, pb, seed):
    rng = np.random.default_rng(seed + 7919)
    x, y, z = _points(pb)
    return torch.stack([_waves(rng, x, y, z) for _ in range(1 if case["physics"] == "advection" else 5)])


def prepare(case, seed):
    pb = _problem_of(case)
    s = Solver(pb, case["physics"], cfl=case["cfl"], gamma=GAMMA, tau_scale=TAU_SCALE, precision=case["precision"],
               flux=case["flux"])
    if case["physics"] == "advection":
        s.set_velocity(*VELOCITY)
    st = dict(kind=case["kind"], steps=case["steps"], solver=s, u0=_initial(case, pb, seed))
    st["out"] = torch.empty_like(st["u0"])
    if case["kind"] == "dirichlet":
        st["g"] = _boundary(case, pb, seed)
    if case["kind"] == "adjoint":
        s.set_adjoint_keep(case["keep"])
        st["every"] = case["every"]
        st["u0"].requires_grad_(True)
        st["gT"] = _cotangent(case, pb, seed)
    if torch.cuda.is_available():
        torch.cuda.synchronize()  # the solver runs on its own stream
    return st


def run(st):
    s, n = st["solver"], st["steps"]
    if st["kind"] == "adjoint":
        uT = dglm_evolve(st["u0"], s, n, every=st["every"])
        (grad,) = torch.autograd.grad(uT, st["u0"], st["gT"])
        return dict(u=uT.detach(), grad=grad)
    s.set_state_device(st["u0"].data_ptr())
    s.set_time(0.0, 0)
    more = {}
    if st["kind"] == "chunk":
        more["dt"] = s.step(n, return_dt=True)
        t, _, tstep, _ = s.time()
        more.update(t=t, tstep=tstep)
    elif st["kind"] == "dirichlet":
        for g in st["g"]:
            s.set_dirichlet_device(g.data_ptr())
            s.step(1)
    else:
        s.step(n)
    s.get_state_device(st["out"].data_ptr())
    return dict(u=st["out"], **more)


def work(case):
    """Per stage: the state and the LSRK register read and written, geometry,
    connectivity, face wave speeds (and the advection velocity) read, and the
    contraction's multiply-adds; per step: the state read for the wave speed.
    An adjoint pass does each forward stage and its transpose once (twice the
    flops; states of the tape written and read, adjoints read and written)."""
    N, K = case["N"], 6 * case["nx"] * case["ny"] * case["nz"]
    nv = 1 if case["physics"] == "advection" else 5
    Np, Nfp = (N + 1) * (N + 2) * (N + 3) // 6, (N + 1) * (N + 2) // 2
    stage_bytes = K * (32 * nv * Np + 8 * 25 + 16 + 32 + (24 * Np if nv == 1 else 0))
    stage_flops = 2 * K * nv * Np * (3 * Np + 4 * Nfp)
    step_bytes = K * (8 * Np * (nv if nv == 5 else 3) + 64)
    n = case["steps"]
    if case["kind"] == "adjoint":
        adj = K * (40 * nv * Np + 16 * nv * 4 * Nfp + 8 * 25 + 16 + 64)
        return dict(bytes=n * (5 * (stage_bytes + adj) + 2 * step_bytes), flops=n * 10 * stage_flops)
    return dict(bytes=n * (5 * stage_bytes + step_bytes), flops=n * 5 * stage_flops)


# ---------------------------------------------------------------------------
# The same pass in plain torch, 64 bits.
# ---------------------------------------------------------------------------
class _Plain:
    def __init__(self, case, pb):
        dev = _device()
        a = pb.arrays
        f = lambda n: torch.as_tensor(np.array(a[n], dtype=np.float64), device=dev)  # noqa: E731
        i = lambda n: torch.as_tensor(np.array(a[n], dtype=np.int64), device=dev).reshape(-1)  # noqa: E731
        self.case, self.K, self.Np, self.Nfp, self.N = case, pb.K, pb.Np, pb.Nfp, pb.N
        self.euler = case["physics"] == "euler"
        self.vmapP, self.vmapF = i("vmapP"), i("vmapF")
        fm = i("Fmask").view(4, pb.Nfp)
        self.vmapM = (torch.arange(pb.K, device=dev)[:, None, None] * pb.Np + fm[None]).reshape(-1)
        self.ops = [f(n).t().contiguous() for n in ("WDr", "WDs", "WDt")] + [f("LIFT").t().contiguous()]
        self.metric = [[f(c + x).view(1, pb.K, 1) for x in "xyz"] for c in "rst"]
        self.n = [f(c).view(1, pb.K * 4, 1) for c in ("nx", "ny", "nz")]
        self.fscale = f("Fscale").view(1, pb.K * 4, 1)
        self.open = None
        if case["kind"] == "dirichlet":
            self.open = torch.as_tensor(_open_faces(pb), device=dev)

    def prim(self, u):
        v = [u[i] / u[0] for i in (1, 2, 3)]
        p = (GAMMA - 1) * (u[4] - 0.5 * u[0] * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]))
        return v, p

    def flux(self, u):
        """The three coordinate fluxes [nvar, ...]."""
        if not self.euler:
            return [c * u for c in VELOCITY]
        v, p = self.prim(u)
        out = []
        for x in range(3):
            F = [u[1 + x]] + [u[i] * v[x] + (p if i == 1 + x else 0.0) for i in (1, 2, 3)] + [(u[4] + p) * v[x]]
            out.append(torch.stack(F))
        return out

    def normal_flux(self, u):
        F = self.flux(u)
        return self.n[0] * F[0] + self.n[1] * F[1] + self.n[2] * F[2]

    def trace(self, u, vmap):
        return torch.index_select(u, 1, vmap).view(u.shape[0], self.K * 4, self.Nfp)

    def speeds(self, u):
        uM = self.trace(u, self.vmapM)
        if not self.euler:
            c = math.sqrt(sum(x * x for x in VELOCITY))
            return torch.full((self.K * 4,), c, dtype=u.dtype, device=u.device)
        v, p = self.prim(uM)
        v2 = (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]).amax(dim=1)
        return torch.sqrt(v2) + torch.sqrt((GAMMA * p / uM[0]).abs().amax(dim=1))

    def rhs(self, u, lam, g):
        K, Np, nv = self.K, self.Np, u.shape[0]
        uM, uP = self.trace(u, self.vmapM), self.trace(u, self.vmapP)
        if self.case["flux"] == "lm":
            tau = (0.25 * TAU_SCALE * (lam + lam[self.vmapF])).view(1, -1, 1)
            ub = 0.5 * (uM + uP)
            if g is not None:
                ub[:, self.open] = g
            fs = self.normal_flux(ub) - tau * (ub - uM)
        else:
            if g is not None:
                uP[:, self.open] = g
            if self.euler:
                c = []
                for q in (uM, uP):
                    v, p = self.prim(q)
                    c.append((self.n[0][0] * v[0] + self.n[1][0] * v[1] + self.n[2][0] * v[2]).abs()
                             + torch.sqrt((GAMMA * p / q[0]).abs()))
                a = torch.maximum(*c)
            else:
                a = (self.n[0] * VELOCITY[0] + self.n[1] * VELOCITY[1] + self.n[2] * VELOCITY[2]).abs()
            fs = 0.5 * (self.normal_flux(uM) + self.normal_flux(uP)) + 0.5 * a * (uM - uP)
        out = -((fs * self.fscale).reshape(nv * K, -1) @ self.ops[3])
        F = [q.view(nv, K, Np) for q in self.flux(u)]
        for d in range(3):
            m = self.metric[d]
            out = out + (m[0] * F[0] + m[1] * F[1] + m[2] * F[2]).reshape(nv * K, Np) @ self.ops[d]
        return out.view(nv, K * Np)

    def step(self, u, k, g=None):
        lam = self.speeds(u)
        dt = self.case["cfl"] / (2 * self.N + 1) / (lam * self.fscale.view(-1)).max()
        for s in range(5):
            k = RKA[s] * k + dt * self.rhs(u, lam, g)
            u = u + RKB[s] * k
        return u, k, dt


def exact(case, seed):
    pb = _problem_of(case)
    P = _Plain(case, pb)
    u0 = _initial(case, pb, seed)
    gs = _boundary(case, pb, seed) if case["kind"] == "dirichlet" else [None] * case["steps"]
    u, k, dts, kept = u0, torch.zeros_like(u0), [], []
    with torch.no_grad():
        for g in gs:
            if case["kind"] == "adjoint":
                kept.append((u, k))
            u, k, dt = P.step(u, k, g)
            dts.append(dt)
    out = dict(u=u)
    if case["kind"] == "chunk":
        dt = torch.stack(dts).cpu().numpy()
        out.update(dt=dt, t=float(sum(dt.tolist())), tstep=case["steps"])
    if case["kind"] == "adjoint":
        ubar, kbar = _cotangent(case, pb, seed), torch.zeros_like(u0)
        for u, k in reversed(kept):
            u, k = u.detach().requires_grad_(True), k.detach().requires_grad_(True)
            u1, k1, _ = P.step(u, k)
            ubar, kbar = torch.autograd.grad((u1, k1), (u, k), (ubar, kbar))
            del u1, k1
        out["grad"] = ubar
    return out
