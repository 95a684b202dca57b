"""Timed cases of the field + LLG path: what a program that uses `mmx` spends its GPU time on.

`listed()` gives the named cases, `draw()` more of the same ranges, `prepare()` the
simulation a program holds before the call, `run()` one pass through the public API and
`exact()` the same result from plain torch in 64 bits.  A pass is one stretch of a
simulation as a script runs it: a number of steps (or one evaluation), then the state read
back.  FP32 simulations keep their state in 32 bits, so their results are handed on as such.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "micromagnetic.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mmx  # noqa: E402

MU0 = 4e-7 * math.pi
# Materials and terms (order of insertion: exchange, DMI, anisotropy, field, demag).
#   soft    permalloy: exchange + demag                        (standard-problem films)
#   field   exchange + in-plane field + demag                  (the published n x n x 1 benchmark)
#   chiral  exchange + interfacial DMI + Ku + field + demag    (skyrmion films)
#   maps    as chiral, D(x,y) and Ku(x,y) per cell, no field   (disordered films, parameter inference)
#   bulk    exchange + bulk DMI + cubic anisotropy + demag     (B20 magnets)
#   stt     exchange + Ku + demag + Zhang-Li current           (racetracks)
MATERIAL = {
    "soft": dict(Ms=8e5, A=1.3e-11, alpha=0.5),
    "field": dict(Ms=8e5, A=1.3e-11, H=(0.0, 0.1 / MU0, 0.0), alpha=0.1),
    "chiral": dict(Ms=5.8e5, A=1.5e-11, Di=3e-3, Ku=8e5, H=(0.0, 0.0, 0.1 / MU0), alpha=0.1),
    "maps": dict(Ms=5.8e5, A=1.5e-11, Di=2.5e-3, Ku=6e5, alpha=0.1),
    "bulk": dict(Ms=8e5, A=1.3e-11, Db=1e-3, Kc=-5e3, alpha=0.1),
    "stt": dict(Ms=5.8e5, A=1.5e-11, Ku=6e5, J=1e12, b=7.2e-11, xi=0.1, alpha=0.2),
}


def listed():
    return [
        # one dm/dt of a small element: programs that step or search on the host call this in a loop
        dict(name="rhs_small", kind="rhs", nx=40, ny=30, nz=1, cell=4.0, pbc="", prec=64, terms="soft", steps=1),
        # 200 x 50 x 1 soft film, Dormand-Prince from a new start state (hysteresis points, switching)
        dict(name="soft_film_rk45", kind="dopri", nx=200, ny=50, nz=1, cell=2.5, pbc="", prec=64, terms="soft",
             steps=20),
        # the published throughput benchmark: n x n x 1, 4 nm cells, 32 bits, Heun
        dict(name="square_film_heun_f32", kind="heun", nx=1000, ny=1000, nz=1, cell=4.0, pbc="", prec=32,
             terms="field", steps=200),
        # a few layers of a skyrmion film with ragged sizes, 64 bits
        dict(name="skyrmion_film_odd", kind="rk4", nx=331, ny=207, nz=3, cell=2.0, pbc="", prec=64, terms="chiral",
             steps=100),
        # 256 x 256 x 32 chiral film, periodic in plane: the large 3-D run, both precisions
        dict(name="chiral_film_f64", kind="rk4", nx=256, ny=256, nz=32, cell=2.0, pbc="xy", prec=64, terms="chiral",
             steps=100),
        dict(name="chiral_film_f32", kind="rk4", nx=256, ny=256, nz=32, cell=2.0, pbc="xy", prec=32, terms="chiral",
             steps=100),
        # 128 x 128 x 8 film with per-cell D and Ku: the forward run of a parameter fit
        dict(name="map_film", kind="rk4", nx=128, ny=128, nz=8, cell=2.0, pbc="", prec=64, terms="maps", steps=200),
        # a thick helimagnet with odd sizes in 32 bits; the state and the energies are recorded
        dict(name="helimagnet_odd_f32", kind="rk4", nx=150, ny=141, nz=51, cell=3.0, pbc="", prec=32, terms="bulk",
             steps=50),
        # domain wall driven along a racetrack (spin-torque term)
        dict(name="racetrack_stt", kind="rk4", nx=600, ny=80, nz=2, cell=2.0, pbc="", prec=64, terms="stt",
             steps=100),
        # uneven parameter sweep and thermal ensemble advanced as one batch, 32 bits
        dict(name="ensemble_f32", kind="batch", nx=96, ny=96, nz=8, cell=2.0, pbc="xy", prec=32, terms="chiral",
             steps=100, members=24),
        # minimum-energy path between two film states
        dict(name="neb_film", kind="neb", nx=64, ny=64, nz=4, cell=2.0, pbc="", prec=64, terms="chiral", steps=50,
             images=14),
        # gradient of a trajectory loss with respect to m0, Ms, D and Ku (backward pass)
        dict(name="adjoint_film", kind="adjoint", nx=96, ny=96, nz=4, cell=2.0, pbc="", prec=64, terms="maps",
             steps=50),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rhs", "dopri", "heun", "rk4", "rk4", "rk4", "rk4", "batch", "neb", "adjoint"])
    prec = rng.choice([64, 32])
    pbc = rng.choice(["", "", "x", "xy"])
    if kind in ("rhs", "dopri"):
        return dict(kind=kind, nx=_spread(rng, 24, 400), ny=_spread(rng, 16, 200), nz=rng.choice([1, 1, 1, 2, 3]),
                    cell=2.5, pbc="", prec=64 if kind == "dopri" else prec, terms="soft",
                    steps=1 if kind == "rhs" else 20)
    if kind == "heun":
        return dict(kind=kind, nx=_spread(rng, 100, 1000), ny=_spread(rng, 100, 1000), nz=1, cell=4.0, pbc="",
                    prec=prec, terms="field", steps=100)
    if kind == "batch":
        return dict(kind=kind, nx=_spread(rng, 40, 120), ny=_spread(rng, 40, 120), nz=rng.randint(4, 10), cell=2.0,
                    pbc="xy", prec=prec, terms="chiral", steps=50, members=rng.randint(6, 24))
    if kind == "neb":
        return dict(kind=kind, nx=_spread(rng, 24, 96), ny=_spread(rng, 24, 96), nz=rng.randint(1, 4), cell=2.0,
                    pbc="", prec=64, terms="chiral", steps=30, images=rng.randint(6, 14))
    if kind == "adjoint":
        return dict(kind=kind, nx=_spread(rng, 24, 100), ny=_spread(rng, 24, 100), nz=rng.randint(1, 4), cell=2.0,
                    pbc=pbc, prec=64, terms="maps", steps=rng.randint(10, 40))
    terms = rng.choice(["chiral", "maps", "bulk", "stt"])
    nx, ny, nz = _spread(rng, 48, 320), _spread(rng, 48, 320), _spread(rng, 1, 48)
    while nx * ny * nz > 1200000:
        nx, ny, nz = max(48, nx * 3 // 4), max(48, ny * 4 // 5), max(1, nz * 4 // 5)
    return dict(kind="rk4", nx=nx, ny=ny, nz=nz, cell=2.0, pbc=pbc, prec=prec, terms=terms, steps=50)


# ---- inputs ------------------------------------------------------------------
_DT = {"soft": 5e-14, "field": 2e-14, "chiral": 1e-14, "maps": 2e-14, "bulk": 2e-14, "stt": 2e-14}


def _state(rng, nx, ny, nz, noise):
    """Smooth random unit vectors (a few Fourier modes) with some noise, 3N values cell by cell."""
    k, j, i = np.meshgrid(np.arange(nz) / max(nz, 4), np.arange(ny) / ny, np.arange(nx) / nx, indexing="ij")
    m = np.zeros((nz, ny, nx, 3))
    for _ in range(6):
        q = rng.integers(-3, 4, 3)
        ph = 2 * np.pi * (q[0] * i + q[1] * j + q[2] * k) + rng.uniform(0, 2 * np.pi)
        m += np.cos(ph)[..., None] * rng.standard_normal(3)
    m += noise * rng.standard_normal(m.shape) + np.array([0.1, 0.05, 0.3])
    m /= np.linalg.norm(m, axis=-1, keepdims=True)
    return m.reshape(-1)


def _map(rng, nx, ny, nz, mean):
    """A correlated random field over (x, y) with 20 % spread, the same in every layer."""
    f = rng.standard_normal((ny, nx))
    ky, kx = np.fft.fftfreq(ny)[:, None], np.fft.rfftfreq(nx)[None, :]
    g = np.fft.irfft2(np.fft.rfft2(f) * np.exp(-0.5 * (kx**2 + ky**2) * (2 * np.pi * 5.0) ** 2), s=(ny, nx))
    g = (g - g.mean()) / g.std()
    return np.tile((mean * (1 + 0.2 * np.clip(g, -3, 3))).reshape(-1), nz)


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    mat = dict(MATERIAL[case["terms"]])
    if case["terms"] == "maps":
        mat["Di"] = _map(rng, nx, ny, nz, mat["Di"])
        mat["Ku"] = _map(rng, nx, ny, nz, mat["Ku"])
    if case["kind"] == "neb":
        # a reversed core moved across the film: the two ends of the path
        y, x = np.meshgrid(np.arange(ny) / ny, np.arange(nx) / nx, indexing="ij")
        ends = []
        for cx in (0.3 + 0.02 * rng.random(), 0.7 - 0.02 * rng.random()):
            r = np.sqrt((x - cx) ** 2 + (y - 0.5) ** 2)
            th = np.pi * np.exp(-((r / 0.12) ** 2))
            ph = np.arctan2(y - 0.5, x - cx)
            v = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], axis=-1)
            v = np.broadcast_to(v, (nz, ny, nx, 3)) + 0.02 * rng.standard_normal((nz, ny, nx, 3))
            ends.append((v / np.linalg.norm(v, axis=-1, keepdims=True)).reshape(-1))
        return mat, ends, None
    noise = 1.0 if case["terms"] == "chiral" else 0.1
    m0 = _state(rng, nx, ny, nz, noise)
    cot = rng.standard_normal(3 * nx * ny * nz) / (nx * ny * nz) if case["kind"] == "adjoint" else None
    return mat, m0, cot


def _member_sizes(case):
    """The sizes belong to the case, the parameters and states of the members to the seed."""
    rng = np.random.default_rng([case["nx"], case["ny"], case["nz"]])
    return [[max(4, int(case[a] * rng.uniform(0.4, 1.4))) for a in ("nx", "ny", "nz")]
            for _ in range(case["members"])]


def _members(case, seed):
    """Uneven members around the case's size: odd ones carry a 300 K stochastic field."""
    rng = np.random.default_rng(seed)
    out = []
    for q, n in enumerate(_member_sizes(case)):
        mat = dict(Ms=rng.uniform(4e5, 1.2e6), A=rng.uniform(5e-12, 2e-11), Di=rng.uniform(1e-3, 4e-3),
                   Ku=rng.uniform(1e5, 1e6), H=MATERIAL["chiral"]["H"], alpha=0.1)
        out.append((n, mat, _state(rng, *n, 0.5), 300.0 if q % 2 else 0.0, int(rng.integers(1 << 30))))
    return out


# ---- the program's side --------------------------------------------------------
_INTEGRATOR = {"rhs": "RungeKutta", "rk4": "RungeKutta", "adjoint": "RungeKutta", "heun": "Heun", "batch": "Heun",
               "dopri": "DormandPrince", "neb": "DormandPrince"}


def _sim(case, n, mat, m0, demag):
    d = case["cell"] * 1e-9
    mesh = mmx.FDMesh(dx=d, dy=d, dz=d, nx=n[0], ny=n[1], nz=n[2], pbc=case["pbc"])
    integ = _INTEGRATOR[case["kind"]]
    sim = mmx.Sim(mesh, integrator=integ, precision=case["prec"])
    sim.driver.alpha = mat["alpha"]
    mmx.set_Ms(sim, mat["Ms"])
    if m0 is not None:
        mmx.init_m0(sim, m0)
    mmx.add_exch(sim, mat["A"])
    if "Di" in mat:
        mmx.add_dmi(sim, mat["Di"], type="interfacial", name="D")
    if "Db" in mat:
        mmx.add_dmi(sim, mat["Db"], type="bulk")
    if "Ku" in mat:
        mmx.add_anis(sim, mat["Ku"], axis=(0, 0, 1), name="Ku")
    if "Kc" in mat:
        mmx.add_cubic_anis(sim, mat["Kc"])
    if "H" in mat:
        mmx.add_zeeman(sim, mat["H"])
    if demag:
        mmx.add_demag(sim)
    if "J" in mat:
        mmx.add_stt(sim, model="zhang_li", J=(mat["J"], 0.0, 0.0), b=mat["b"], xi=mat["xi"])
    if integ in ("RungeKutta", "Heun"):
        mmx.set_driver(sim, integrator=integ, step=_DT[case["terms"]])
    return sim


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        sims = []
        for n, mat, m0, temp, s in _members(case, seed):
            sim = _sim(case, n, mat, m0, demag=False)
            if temp:
                mmx.add_thermal_noise(sim, temp, seed=s)
            sims.append(sim)
        return dict(case=case, sims=sims, batch=mmx.Batch(sims))
    mat, m0, cot = _inputs(case, seed)
    n = (case["nx"], case["ny"], case["nz"])
    if kind == "neb":
        sim = _sim(case, n, mat, m0[0], demag=True)
        return dict(case=case, sim=sim, neb=mmx.NEB(sim, m0, [case["images"]], spring_constant=1e5))
    sim = _sim(case, n, mat, m0, demag=kind != "adjoint")
    return dict(case=case, sim=sim, m0=m0, cot=cot)


def _own(case, a):
    return a.astype(np.float32) if case["prec"] == 32 else a


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "batch":
        state["batch"].advance(case["steps"])
        return [_own(case, s.spin) for s in state["sims"]]
    if kind == "neb":
        state["neb"].advance(case["steps"])
        return {"images": state["neb"].spin, "energy": state["neb"].energy}
    sim = state["sim"]
    if kind == "rhs":
        return _own(case, mmx.llg_rhs(sim, state["m0"]))
    if kind == "dopri":
        mmx.init_m0(sim, state["m0"])
        mmx.set_driver(sim, integrator="DormandPrince", tol=1e-6)
        mmx.run_until(sim, case["steps"] * 5e-13)
        return sim.spin
    if kind == "adjoint":
        mmx.init_m0(sim, state["m0"])
        m, pullback = mmx.rk4_trajectory_rrule(sim, case["steps"], every=20)
        return {"m": m, "grad": pullback(state["cot"])}
    mmx.run_step(sim, n=case["steps"])
    if case["terms"] == "bulk":
        return {"m": _own(case, sim.spin), "energy": _own(case, mmx.compute_system_energy(sim))}
    return _own(case, sim.spin)


# ---- what a pass cannot do without ---------------------------------------------
_EVALS = {"rhs": 1, "heun": 2, "rk4": 4, "batch": 2, "neb": 3, "adjoint": 12, "dopri": 7}


def _pad(n):
    return 1 if n == 1 else 2 * n


def work(case):
    """Per evaluation: m and mu0 Ms read, per-cell parameters read, a 3-vector written, and
    with demag the six k-space tensor components read once (one octant) and six transforms of
    the zero-padded mesh; per step the stage vectors that the scheme combines."""
    w = case["prec"] // 8
    kind, steps = case["kind"], case["steps"]
    N = case["nx"] * case["ny"] * case["nz"]
    evals = steps * _EVALS[kind]
    if kind == "batch":
        N = sum(n[0] * n[1] * n[2] for n in _member_sizes(case))
    if kind == "neb":
        N *= case["images"]
    maps = 2 if case["terms"] == "maps" else 0
    nbytes = w * N * (7 + maps) * evals
    flops = 150.0 * N * evals
    nbytes += {"rk4": 30, "heun": 9, "batch": 9, "dopri": 75, "neb": 30, "adjoint": 60, "rhs": 0}[kind] * w * N * steps
    if kind not in ("batch", "adjoint"):
        P = [_pad(case[a]) for a in ("nx", "ny", "nz")]
        total = float(P[0] * P[1] * P[2])
        many = case["images"] if kind == "neb" else 1
        nbytes += 6 * w * (P[0] // 2 + 1) * (P[1] // 2 + 1) * (P[2] // 2 + 1) * evals
        flops += many * evals * (6 * 2.5 * total * math.log2(max(total, 2)) + 15 * total)
    return {"bytes": float(nbytes), "flops": float(flops)}


# ---- the same in plain torch, 64 bits --------------------------------------------
def _newell(n, d, dev):
    """Demag tensor (xx, yy, zz, xy, xz, yz) on displacements -(n-1)..(n-1) (Newell, Williams and
    Dunlop 1993); the point dipole beyond 60 cell edges."""
    def grid(q):
        ax = [torch.arange(-m, m + 1, dtype=torch.float64, device=dev) * q for m in n]
        return torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")[::-1]

    def safe(num, den):
        return torch.where(den == 0, torch.zeros_like(num), num / torch.where(den == 0, torch.ones_like(den), den))

    def f(x, y, z):
        x2, y2, z2 = x * x, y * y, z * z
        R = torch.sqrt(x2 + y2 + z2)
        v = (2 * x2 - y2 - z2) * R / 6 - x * y * z * torch.atan(safe(y * z, x * R))
        v = v + 0.5 * y * (z2 - x2) * torch.asinh(safe(y, torch.sqrt(x2 + z2)))
        return v + 0.5 * z * (y2 - x2) * torch.asinh(safe(z, torch.sqrt(x2 + y2)))

    def g(x, y, z):
        x2, y2, z2 = x * x, y * y, z * z
        R = torch.sqrt(x2 + y2 + z2)
        v = -x * y * R / 3 - z2 * z * torch.atan(safe(x * y, z * R)) / 6
        v = v - 0.5 * y2 * z * torch.atan(safe(x * z, y * R)) - 0.5 * x2 * z * torch.atan(safe(y * z, x * R))
        v = v + x * y * z * torch.asinh(safe(z, torch.sqrt(x2 + y2)))
        v = v + y * (3 * z2 - y2) * torch.asinh(safe(x, torch.sqrt(y2 + z2))) / 6
        return v + x * (3 * z2 - x2) * torch.asinh(safe(y, torch.sqrt(x2 + z2))) / 6

    X, Y, Z = grid(1.0)  # cubic cells, in units of the edge
    far = torch.sqrt(X * X + Y * Y + Z * Z) > 60

    def second(a, dim):
        lo, mid, hi = (a.narrow(dim, s, a.shape[dim] - 2) for s in (0, 1, 2))
        return 2 * mid - lo - hi

    def near(fn, x, y, z):
        v = fn(x, y, z)
        for dim in range(3):
            v = second(v, dim)
        return v / (4 * math.pi)

    def dipole(a, b, x, y, z):
        R2 = x * x + y * y + z * z
        R2 = torch.where(R2 == 0, torch.ones_like(R2), R2)
        v = -3 * a * b / (R2 * R2 * torch.sqrt(R2))
        if a is b:
            v = v + 1 / (R2 * torch.sqrt(R2))
        return v / (4 * math.pi)

    inner = (slice(1, -1),) * 3
    out = []
    for fn, a in ((f, (X, Y, Z)), (f, (Y, X, Z)), (f, (Z, Y, X)), (g, (X, Y, Z)), (g, (X, Z, Y)), (g, (Y, Z, X))):
        v = near(fn, *a)
        pair = (a[0], a[0]) if fn is f else (a[0], a[1])
        w = dipole(*pair, X, Y, Z)[inner]
        out.append(torch.where(far[inner], w, v))
    return out


class _Reference:
    """H_eff and dm/dt of one case in torch; m is (3, nz, ny, nx)."""

    def __init__(self, case, n, mat, demag, dev):
        self.n, self.mat, self.d = n, mat, case["cell"] * 1e-9
        self.pbc, self.dev = case["pbc"], dev
        self.mus = MU0 * mat["Ms"]
        self.par = {k: self._cells(mat[k]) for k in ("Di", "Ku") if k in mat}
        self.K = None
        if demag:
            self.P = [1 if q == 1 else 2 * q for q in n]
            self.K = []
            for t in _newell(n, self.d, dev):
                pad = torch.zeros(self.P[2], self.P[1], self.P[0], dtype=torch.float64, device=dev)
                idx = [torch.arange(-(q - 1), q, device=dev) % p for q, p in zip(n, self.P)]
                pad[idx[2][:, None, None], idx[1][None, :, None], idx[0][None, None, :]] = t
                self.K.append(torch.fft.rfftn(pad))

    def _cells(self, v):
        v = torch.as_tensor(v, dtype=torch.float64, device=self.dev)
        return v if v.dim() == 0 else v.reshape(self.n[2], self.n[1], self.n[0])

    def vec(self, a):
        a = torch.as_tensor(a, dtype=torch.float64, device=self.dev)
        return a.reshape(self.n[2], self.n[1], self.n[0], 3).permute(3, 0, 1, 2).contiguous()

    @staticmethod
    def flat(m):
        return m.permute(1, 2, 3, 0).reshape(-1).cpu().numpy()

    def nb(self, a, axis, step):
        """Neighbour values along axis (0 x, 1 y, 2 z) and a 0/1 mask of those that exist."""
        dim = a.dim() - 1 - axis
        v = torch.roll(a, -step, dim)
        ok = torch.ones(self.n[2], self.n[1], self.n[0], dtype=torch.float64, device=self.dev)
        if "xyz"[axis] not in self.pbc:
            ok.narrow(2 - axis, ok.shape[2 - axis] - 1 if step > 0 else 0, 1).zero_()
        return v, ok

    def local(self, m, par, mus):
        f = torch.zeros_like(m)
        c = 2 * self.mat["A"] / self.d**2
        for axis in range(3):
            for step in (-1, 1):
                v, ok = self.nb(m, axis, step)
                f = f + c * ok * (v - m)
                e = [0.0, 0.0, 0.0]
                if "Db" in self.mat:
                    e[axis] = -step * self.mat["Db"] / self.d
                    f = f + ok * self.cross(e, v)
                if "Di" in par and axis < 2:
                    D = par["Di"]
                    if D.dim():
                        Dn = self.nb(D, axis, step)[0]
                        D = 2 * D * Dn / (D + Dn)
                    e = [0.0, -step / self.d, 0.0] if axis == 0 else [step / self.d, 0.0, 0.0]
                    f = f + ok * D * self.cross(e, v)
        if "Ku" in par:
            f = f + torch.stack([torch.zeros_like(m[0]), torch.zeros_like(m[0]), 2 * par["Ku"] * m[2]])
        if "Kc" in self.mat:
            f = f + 4 * self.mat["Kc"] * m**3
        h = f / mus
        if "H" in self.mat:
            h = h + torch.tensor(self.mat["H"], dtype=torch.float64, device=self.dev)[:, None, None, None]
        return h

    @staticmethod
    def cross(a, b):
        return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])

    def demag(self, m):
        F = torch.fft.rfftn(self.mus * m, s=(self.P[2], self.P[1], self.P[0]), dim=(1, 2, 3))
        xx, yy, zz, xy, xz, yz = self.K
        G = torch.stack([xx * F[0] + xy * F[1] + xz * F[2], xy * F[0] + yy * F[1] + yz * F[2],
                         xz * F[0] + yz * F[1] + zz * F[2]])
        h = torch.fft.irfftn(G, s=(self.P[2], self.P[1], self.P[0]), dim=(1, 2, 3))
        return -h[:, : self.n[2], : self.n[1], : self.n[0]] / MU0

    def stt(self, m):
        """Zhang-Li: (1/gamma) (m x (u.grad)m + xi (u.grad)m), one-sided at the ends."""
        lo, okl = self.nb(m, 0, -1)
        hi, okh = self.nb(m, 0, 1)
        both = okl * okh
        g = (okh * hi + (1 - okh) * m - okl * lo - (1 - okl) * m) * (both / (2 * self.d) + (1 - both) / self.d)
        g = g * self.mat["J"] * self.mat["b"] / 2.21e5
        return self.cross(m, g) + self.mat["xi"] * g

    def rhs(self, m, par=None, mus=None):
        h = self.local(m, par or self.par, self.mus if mus is None else mus)
        if self.K is not None:
            h = h + self.demag(m)
        if "J" in self.mat:
            h = h + self.stt(m)
        al = self.mat["alpha"]
        p = (m * m).sum(0) * h - (m * h).sum(0) * m
        return -2.21e5 / (1 + al * al) * (self.cross(m, p) - al * p)

    def energy(self, m):
        """Exchange, bulk DMI, cubic and demag energies (J) of the `bulk` material."""
        V, out, full = self.d**3, [], self.mat
        for keep in ("A", "Db"):
            self.mat = {"A": full["A"] if keep == "A" else 0.0}
            if keep == "Db":
                self.mat["Db"] = full["Db"]
            out.append(float(-0.5 * V * self.mus * (m * self.local(m, {}, self.mus)).sum()))
        self.mat = full
        out.append(float(-full["Kc"] * V * (m**4).sum()))
        out.append(float(-0.5 * V * self.mus * (m * self.demag(m)).sum()))
        return np.array(out)

    def rk4(self, m, h, par=None, mus=None):
        k1 = self.rhs(m, par, mus)
        k2 = self.rhs(m + 0.5 * h * k1, par, mus)
        k3 = self.rhs(m + 0.5 * h * k2, par, mus)
        k4 = self.rhs(m + h * k3, par, mus)
        return self.unit(m + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4))

    def heun(self, m, h):
        k1 = self.rhs(m)
        k2 = self.rhs(m + h * k1)
        return self.unit(m + 0.5 * h * (k1 + k2))

    @staticmethod
    def unit(m):
        return m / torch.sqrt((m * m).sum(0))

    def dopri(self, m, t_end, tol):
        """Dormand-Prince 5(4), the step control of an AdaptiveRK run to t_end."""
        A = [[1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
             [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
             [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656],
             [35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]]
        E = [71 / 57600, 0.0, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40]
        t = 0.0
        r = float(self.rhs(m).abs().max()) / (0.824 * tol**0.2)
        nxt = min(1e-12, 0.001 / r if 1e-12 * r > 0.001 else 1e-12)
        while t < t_end:
            if nxt + t > t_end:
                nxt = t_end - t
            h = nxt
            while True:
                k = [self.rhs(m)]
                for row in A:
                    y = m + h * sum(a * q for a, q in zip(row, k))
                    y = self.unit(y) if row is A[-1] else y
                    k.append(self.rhs(y))
                e = sum(a * q for a, q in zip(E, k))
                err = float((e.abs() / (1 + y.abs())).max()) * h / tol
                if err <= 1:
                    break
                h *= min(5.0, max(0.2, 0.824 * (1 / err) ** 0.25))
            t, m = t + h, y
            nxt = h * min(5.0, max(0.2, 0.824 * (1 / err) ** 0.2))
        return m


def exact(case, seed):
    kind, h = case["kind"], _DT[case["terms"]]
    if kind == "neb":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    n = (case["nx"], case["ny"], case["nz"])
    if dev == "cpu" and n[0] * n[1] * n[2] * case["steps"] > 4000000:
        return None
    if kind == "batch":  # the stochastic members have no such value
        out = []
        for size, mat, m0, temp, _ in _members(case, seed):
            ref = None if temp else _Reference(case, size, mat, False, dev)
            m = ref.vec(m0) if ref else None
            for _ in range(case["steps"] if ref else 0):
                m = ref.heun(m, h)
            out.append(ref.flat(m) if ref else None)
        return out
    mat, m0, cot = _inputs(case, seed)
    ref = _Reference(case, n, mat, kind != "adjoint", dev)
    m = ref.vec(m0)
    if kind == "rhs":
        return ref.flat(ref.rhs(m))
    m = ref.unit(m)
    if kind == "dopri":
        return ref.flat(ref.dopri(m, case["steps"] * 5e-13, 1e-6))
    if kind == "adjoint":
        return _exact_gradient(case, ref, m, ref.vec(cot), h)
    for _ in range(case["steps"]):
        m = ref.heun(m, h) if kind == "heun" else ref.rk4(m, h)
    if case["terms"] == "bulk":
        return {"m": ref.flat(m), "energy": ref.energy(m)}
    return ref.flat(m)


def _exact_gradient(case, ref, m, lam, h):
    """The trajectory's pull-back step by step through torch.autograd."""
    states = [m]
    for _ in range(case["steps"]):
        states.append(ref.rk4(states[-1], h))
    mus = torch.full_like(m[0], ref.mus)
    leaves = {"Ku": ref.par["Ku"], "D": ref.par["Di"], "Ms": mus}
    grads = {k: torch.zeros_like(v) for k, v in leaves.items()}
    for y in reversed(states[:-1]):
        p = {k: v.detach().clone().requires_grad_(True) for k, v in leaves.items()}
        y = y.detach().clone().requires_grad_(True)
        out = ref.rk4(y, h, {"Ku": p["Ku"], "Di": p["D"]}, p["Ms"])
        got = torch.autograd.grad(out, [y] + [p[k] for k in leaves], lam)
        lam = got[0]
        for k, g in zip(leaves, got[1:]):
            grads[k] = grads[k] + g
    g = {k: v.reshape(-1).cpu().numpy() for k, v in grads.items()}
    g["Ms"] = g["Ms"] * MU0
    g["m0"] = ref.flat(lam)
    return {"m": ref.flat(states[-1]), "grad": g}
