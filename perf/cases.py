"""The calls whose speed matters to a user of this framework, with their inputs and exact results.

A case is one pass through the public entry points (``GpuDomain.step``, ``GpuBatch.step``,
``GpuDomain.adjoint``).  Four families cover what a user runs:

* ``wave``: ideal MHD alone on a periodic box (RK2 or RK4), from grids of a few thousand cells,
  where a step is a handful of short launches, to 2048 x 2048;
* ``arcade``: the solar arcade, ideal MHD with field-aligned thermal conduction (with or without
  flux saturation, Euler or RK2 subcycles) and radiative losses, with a fixed lower and an open
  upper side;
* ``plasma``: one two-fluid plasma expansion, or a batch of them of uneven sizes;
* ``adjoint``: the gradient of a scalar of the final state through several steps, of the wave
  (in plane, RK2) or of the heated arcade (conduction, radiation, parametrised heating).

A pass of the ideal-MHD families starts from the same initial condition every time: the program
keeps it on the device, writes it into the domain's live grids (``spruce_gpu_device_grid``, on the
domain's own stream), propagates and runs its steps, as a parameter study or an optimisation loop
does.  The two-fluid families step on from where the last pass ended.

All numbers are binary64.  ``exact`` restates the same equations in whole-grid torch operations.
"""
from __future__ import annotations

import ctypes
import math
from typing import Dict, List, Optional

import numpy as np
import torch

from spruce_amd.gpu import GpuBatch, GpuDomain, lib
from spruce_amd.spec import DomainSpec

PERIODIC, OPEN, FIXED, OPEN_UCNP = 0, 1, 2, 5
EULER, RK2, RK4 = 0, 1, 2
K_B = 1.3807e-16
M_PROTON = 1.6726e-24
M_SR = 1.455e-22
M_ELECTRON = 9.1094e-28
E_CHARGE = 4.80320425e-10
C_LIGHT = 29979245800.0
GAMMA = 1.6666666666666667
MHD_EVOLVED = ("rho", "mom_x", "mom_y", "mom_z", "thermal_energy", "bi_x", "bi_y", "bi_z")
TF_EVOLVED = ("i_rho", "e_rho", "i_mom_x", "i_mom_y", "e_mom_x", "e_mom_y", "i_thermal_energy", "e_thermal_energy",
              "E_x", "E_y", "E_z", "bi_x", "bi_y", "bi_z")
BATCH_EDGES = (128, 192, 256, 384, 512)   # edges of the batched workload's members


def listed() -> List[dict]:
    return [
        # a small box as in a first test or a course: launches and their gaps are the whole step
        dict(name="wave_64x48", family="wave", nx=64, ny=48, integrator=RK2, out_of_plane=False, steps=50),
        # the plain workload of the framework's own benchmark
        dict(name="wave_256", family="wave", nx=256, ny=256, integrator=RK2, out_of_plane=False, steps=50),
        # an ordinary run at odd sizes, with all three components and the four-stage integrator
        dict(name="wave_515x389_rk4", family="wave", nx=515, ny=389, integrator=RK4, out_of_plane=True, steps=10),
        # a large plain run: the stage kernel's throughput
        dict(name="wave_2048", family="wave", nx=2048, ny=2048, integrator=RK2, out_of_plane=False, steps=4),
        # a small ragged arcade, as one looks at before a production run
        dict(name="arcade_133x197", family="arcade", nx=133, ny=197, saturation=False, tc_integrator="euler", steps=10),
        # the arcade at the size its physics was set up for
        dict(name="arcade_512x1024", family="arcade", nx=512, ny=1024, saturation=False, tc_integrator="euler", steps=5),
        # the same physics with flux saturation and second-order subcycles, at an odd size
        dict(name="arcade_700x1301_sat", family="arcade", nx=700, ny=1301, saturation=True, tc_integrator="rk2", steps=3),
        # the headline workload
        dict(name="arcade_2048", family="arcade", nx=2048, ny=2048, saturation=False, tc_integrator="euler", steps=4),
        # one two-fluid expansion
        dict(name="plasma_192", family="plasma", members=1, nx=192, ny=192, steps=20),
        # a study over many expansions of uneven sizes, advanced together
        dict(name="plasma_batch_16", family="plasma", members=16, nx=0, ny=0, steps=10),
        # gradient through the plain step
        dict(name="adjoint_wave_256", family="adjoint", nx=256, ny=256, arcade=False, checkpoint=10, steps=20),
        # gradient of the heated arcade with respect to its state and heating coefficients
        dict(name="adjoint_arcade_384x512", family="adjoint", nx=384, ny=512, arcade=True, checkpoint=2, steps=3),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(("wave", "wave", "arcade", "arcade", "plasma", "adjoint"))
    if kind == "wave":
        nx, ny = _log(rng, 40, 2048), _log(rng, 40, 2048)
        integ = rng.choice((RK2, RK2, RK4))
        steps = max(2, min(50, 16_000_000 // (nx * ny * (2 if integ == RK4 else 1))))
        return dict(family="wave", nx=nx, ny=ny, integrator=integ, out_of_plane=rng.random() < 0.5, steps=steps)
    if kind == "arcade":
        sat, integ = rng.random() < 0.3, rng.choice(("euler", "euler", "rk2"))
        top = 2048 if not sat and integ == "euler" else 1024   # the others cost twice to four times as much a cell
        nx, ny = _log(rng, 64, top), _log(rng, 128, top)
        return dict(family="arcade", nx=nx, ny=ny, saturation=sat, tc_integrator=integ,
                    steps=2 if nx * ny > 1_000_000 else rng.randint(3, 6))
    if kind == "plasma":
        if rng.random() < 0.5:
            return dict(family="plasma", members=1, nx=_log(rng, 64, 512), ny=_log(rng, 64, 512), steps=rng.randint(6, 15))
        return dict(family="plasma", members=rng.randint(2, 16), nx=0, ny=0, steps=rng.randint(4, 9))
    arcade = rng.random() < 0.5
    if arcade:
        return dict(family="adjoint", nx=_log(rng, 64, 384), ny=_log(rng, 128, 512), arcade=True,
                    checkpoint=rng.randint(1, 3), steps=rng.randint(2, 3))
    return dict(family="adjoint", nx=_log(rng, 64, 320), ny=_log(rng, 64, 320), arcade=False, checkpoint=rng.randint(3, 9),
                steps=rng.randint(6, 18))


# --------------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------------

def _mesh(dx: np.ndarray, dy: np.ndarray) -> Dict[str, np.ndarray]:
    nx, ny = len(dx), len(dy)
    px, py = np.cumsum(dx) - 0.5 * dx, np.cumsum(dy) - 0.5 * dy
    full = lambda a, ax: np.ascontiguousarray(np.broadcast_to(a[:, None] if ax == 0 else a[None, :], (nx, ny)))  # noqa: E731
    return {"d_x": full(dx, 0), "d_y": full(dy, 1), "pos_x": full(px, 0), "pos_y": full(py, 1)}


def _wave_spec(case: dict, seed: int) -> DomainSpec:
    """Noisy density and temperature with a sheared flow and field (periodic box)."""
    nx, ny = case["nx"], case["ny"]
    rng = np.random.default_rng(seed)
    noise = lambda a: a * (2.0 * rng.random((nx, ny)) - 1.0)  # noqa: E731
    d, rho0, t0, v0, b0 = 1e7, 1e-15, 1e6, 1e7, 1.0
    x, y = ((np.arange(nx) + 0.5) / nx)[:, None], ((np.arange(ny) + 0.5) / ny)[None, :]
    z = np.zeros((nx, ny))
    rho = rho0 * (1.0 + noise(0.05))
    g = _mesh(np.full(nx, d), np.full(ny, d))
    g.update(rho=rho, temp=t0 * (1.0 + noise(0.02)), mom_x=-rho * v0 * np.sin(2 * np.pi * y) * (1.0 + noise(0.01)),
             mom_y=rho * v0 * np.sin(2 * np.pi * x) * (1.0 + noise(0.01)), mom_z=z,
             bi_x=-b0 * np.sin(2 * np.pi * y) + z, bi_y=b0 * np.sin(4 * np.pi * x) + z, bi_z=z,
             be_x=z, be_y=z, be_z=z, grav_x=z, grav_y=z)
    if case.get("out_of_plane", True):
        g.update(mom_z=rho * v0 * noise(0.1), bi_z=b0 * (0.5 + noise(0.1)))
    if case["family"] == "adjoint":   # off the limiter's exact ties, where the gradient is not unique
        g.update(bi_x=g["bi_x"] + noise(0.01), bi_y=g["bi_y"] + noise(0.01))
    return DomainSpec(nx, ny, (PERIODIC,) * 4, case.get("integrator", RK2), 0.2, 1.0, 1.0, 1e-12, 0.0, 1.0, M_PROTON, GAMMA,
                      "ideal_mhd", grids={k: np.ascontiguousarray(v, np.float64) for k, v in g.items()})


def _arcade_spec(case: dict, seed: int) -> DomainSpec:
    """Stratified atmosphere in a line-dipole field on a mesh stretched upwards, 1% noise on it."""
    nx, ny = case["nx"], case["ny"]
    rng = np.random.default_rng(seed)
    noise = lambda a: a * (2.0 * rng.random((nx, ny)) - 1.0)  # noqa: E731
    # tall meshes stretch less: ten scale heights up the density is at its floor and conduction unstable
    dx, dy = np.full(nx, 5e6), 5e6 * (1.0005 if ny > 512 else 1.002) ** np.arange(ny)
    x, y = (np.arange(nx) + 0.5) * 5e6, np.cumsum(dy) - 0.5 * dy
    depth, lx, grav = 6.4e8, nx * 5e6, -2.74e4
    zz = (x[:, None] - 0.5 * lx) + 1j * (y[None, :] + depth)
    b = -10.0 * depth * depth / zz ** 2
    T1 = 2e4 + (1e6 - 2e4) * 0.5 * (1.0 + np.tanh((y - 2.0e8) / 4.0e7))
    lnp = np.concatenate([[0.0], np.cumsum(-M_PROTON * -grav * np.diff(y) / (2 * K_B) * 0.5 * (1 / T1[:-1] + 1 / T1[1:]))])
    n1 = 3e11 * 2e4 / T1 * np.exp(lnp)
    z = np.zeros((nx, ny))
    g = _mesh(dx, dy)
    g.update(rho=M_PROTON * n1[None, :] * (1.0 + noise(0.01)), temp=T1[None, :] * (1.0 + noise(0.01)), mom_x=z, mom_y=z,
             mom_z=z, bi_x=z, bi_y=z, bi_z=z, be_x=b.real, be_y=-b.imag, be_z=z, grav_x=z, grav_y=z + grav)
    if case["family"] == "adjoint":   # off the limiter's exact ties, where the gradient is not unique
        v = 1e5 * g["rho"]
        g.update(mom_x=v * noise(1.0), mom_y=v * noise(1.0), mom_z=v * noise(1.0), bi_x=noise(0.01), bi_y=noise(0.01),
                 bi_z=noise(0.01))
    modules = [("thermal_conduction", [("flux_saturation", "true" if case.get("saturation") else "false"),
                                       ("epsilon", "0.5"), ("dt_subcycle_min", "1e-6"),
                                       ("time_integrator", case.get("tc_integrator", "euler"))]),
               ("radiative_losses", [("cutoff_ramp", "2e4"), ("cutoff_temp", "3e4"), ("epsilon", "0.5"),
                                     ("time_integrator", "euler")])]
    if case["family"] == "adjoint":
        modules.append(("parametric_heating", [("num_basis", "16")] +
                        [("coeff_%d" % k, repr(float(t))) for k, t in enumerate(_theta())]))
    return DomainSpec(nx, ny, (PERIODIC, PERIODIC, FIXED, OPEN), RK2, 0.2, 1.0, 1e4, 1e-8, 0.0, 1.0, M_PROTON, GAMMA,
                      "ideal_mhd", modules=modules, grids={k: np.ascontiguousarray(v, np.float64) for k, v in g.items()})


def _theta() -> np.ndarray:
    return 1e-4 * (1.0 + 0.5 * np.sin(np.arange(16)))


def _plasma_specs(case: dict, seed: int) -> List[DomainSpec]:
    """Gaussian plasmas expanding into a thin background; a batch draws each member's size and peak."""
    rng = np.random.default_rng(seed)
    sizes = np.random.default_rng(7)   # a batch's sizes belong to the case, its plasmas to the seed
    out = []
    for _ in range(case["members"]):
        e = int(sizes.choice(BATCH_EDGES))
        nx, ny = (case["nx"], case["ny"]) if case["members"] == 1 else (e, e)
        sigma, peak = 0.05 + 0.1 * rng.random(), 1e9 + 9e9 * rng.random()
        te = 50.0 + 150.0 * rng.random()
        L = 8 * sigma
        x, y = (np.arange(nx) + 0.5) * L / nx - 0.5 * L, (np.arange(ny) + 0.5) * L / ny - 0.5 * L
        n = peak * np.exp(-(x[:, None] ** 2 + y[None, :] ** 2) / (2 * sigma * sigma)) + 1e-4 * peak
        n = n * (1.0 + 0.01 * (2 * rng.random((nx, ny)) - 1))
        z = np.zeros((nx, ny))
        g = _mesh(np.full(nx, L / nx), np.full(ny, L / ny))
        g.update({k: z for k in ("i_mom_x", "i_mom_y", "e_mom_x", "e_mom_y", "bi_x", "bi_y", "bi_z", "be_x", "be_y", "be_z",
                                 "E_x", "E_y", "E_z", "grav_x", "grav_y")})
        g.update(i_rho=n * M_SR, e_rho=n * M_ELECTRON, i_temp=z + 1.0, e_temp=z + te)
        out.append(DomainSpec(nx, ny, (OPEN_UCNP,) * 4, RK2, 0.2, 1e2, 1e-3, 1e-30, 0.0, 1.0, M_SR, GAMMA, "ideal_2F",
                              equation_set_options=[("use_sub_cycling", "false"), ("remove_curl_terms", "true")],
                              grids={k: np.ascontiguousarray(v, np.float64) for k, v in g.items()}))
    return out


def _mhd_spec(case: dict, seed: int) -> DomainSpec:
    arcade = case["family"] == "arcade" or case.get("arcade", False)
    return _arcade_spec(case, seed) if arcade else _wave_spec(case, seed)


def _loss_seed(case: dict, spec: DomainSpec, seed: int) -> np.ndarray:
    """dJ/d(final evolved grids) of a smooth random functional, each grid scaled by its own magnitude."""
    rng = np.random.default_rng(seed + 1_000_003)
    rho, T = spec.grids["rho"], spec.grids["temp"]
    scale = [rho, 1e6 * rho, 1e6 * rho, 1e6 * rho, 3 * K_B * T * rho / M_PROTON, 1.0, 1.0, 1.0]
    return np.stack([rng.standard_normal((case["nx"], case["ny"])) / s for s in scale])


# --------------------------------------------------------------------------------------------
# A pass
# --------------------------------------------------------------------------------------------

class _DeviceGrid:
    """A live grid of a domain as an array on the device, valid until the domain's next step; a tensor
    made from it keeps the domain, which owns the memory."""

    def __init__(self, dom: GpuDomain, name: str):
        self.owner = dom
        p = ctypes.POINTER(ctypes.c_double)()
        if lib().spruce_gpu_device_grid(dom.h, name.encode(), ctypes.byref(p)) < 0:
            raise RuntimeError(lib().spruce_gpu_last_error().decode())
        self.__cuda_array_interface__ = {"shape": (dom.spec.xdim, dom.spec.ydim), "typestr": "<f8", "version": 3,
                                         "data": (ctypes.cast(p, ctypes.c_void_p).value, False), "strides": None}


def _grids(dom: GpuDomain, names) -> Dict[str, torch.Tensor]:
    return {n: torch.as_tensor(_DeviceGrid(dom, n), device="cuda") for n in names}


class _Start:
    """A domain's initial condition kept on the device, and the stream its grids are written on."""

    def __init__(self, dom: GpuDomain):
        self.stream = torch.cuda.ExternalStream(dom.stream())
        self.grids = {k: v.clone() for k, v in _grids(dom, MHD_EVOLVED).items()}

    def restore(self, dom: GpuDomain) -> None:
        with torch.cuda.stream(self.stream):
            for k, v in _grids(dom, MHD_EVOLVED).items():
                v.copy_(self.grids[k])
        dom.propagate()


def prepare(case: dict, seed: int) -> dict:
    if case["family"] == "plasma":
        domains = [GpuDomain(s) for s in _plasma_specs(case, seed)]
        return {"case": case, "dom": domains[0]} if len(domains) == 1 else {"case": case, "batch": GpuBatch(domains)}
    spec = _mhd_spec(case, seed)
    dom = GpuDomain(spec)
    state = {"case": case, "dom": dom, "start": _Start(dom)}
    if case["family"] == "adjoint":
        state["seed"] = _loss_seed(case, spec, seed)
    spec.grids.clear()
    return state


def run(state: dict):
    case = state["case"]
    if case["family"] == "plasma":
        if "batch" in state:
            dts = state["batch"].step(case["steps"])
            return {"dt": dts, "members": [torch.stack(list(_grids(d, TF_EVOLVED[:10]).values()))
                                           for d in state["batch"].domains]}
        dts = state["dom"].step(case["steps"])
        return {"dt": dts, **_grids(state["dom"], TF_EVOLVED[:10])}
    dom = state["dom"]
    state["start"].restore(dom)
    if case["family"] == "adjoint":
        grad, dts = dom.adjoint(case["steps"], case["checkpoint"], state["seed"])
        out = {"dt": dts, "grad": dict(zip(MHD_EVOLVED, grad)), **_grids(dom, MHD_EVOLVED)}
        if case["arcade"]:
            out["grad_theta"] = dom.adjoint_params()
        return out
    dts = dom.step(case["steps"])
    return {"dt": dts, **_grids(dom, MHD_EVOLVED)}


# --------------------------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------------------------

def work(case: dict) -> dict:
    """Bytes: per step, the evolved and static grids read once and the evolved grids written once (a
    step needs the whole grid's smallest time scale, so steps cannot share a pass over memory); an
    adjoint does that for the step and for its reverse.  Operations: the stencil's per cell and
    stage, and the conduction update's per subcycle at a typical count."""
    steps = case["steps"]
    if case["family"] == "plasma":
        sizes = np.random.default_rng(7)
        cells = sum(int(sizes.choice(BATCH_EDGES)) ** 2 for _ in range(case["members"]))
        cells = case["nx"] * case["ny"] if case["members"] == 1 else cells
        return {"bytes": cells * steps * (14 + 2 + 14) * 8, "flops": cells * steps * 2 * 500}
    cells = case["nx"] * case["ny"]
    stages = 4 if case.get("integrator", RK2) == RK4 else 2
    flops = 650 * stages
    if case["family"] == "arcade" or case.get("arcade"):
        flops += 130 * 30 * (2 if case.get("tc_integrator") == "rk2" else 1)
    passes = 3 if case["family"] == "adjoint" else 1   # forward, recompute, reverse
    return {"bytes": cells * steps * (8 + 5 + 8) * 8 * (2 if passes == 3 else 1), "flops": cells * steps * flops * passes}


def tolerance(case: dict):
    """Binary64 with a few hundred to a few thousand roundings along a chain.  Against ``exact``: the
    wave and the plasma 1e-15 .. 6e-15; an arcade's momenta and induced field, differences of much
    larger terms, up to 3e-11 at 2048 x 2048; gradients, which sum over each cell's neighbours in no
    fixed order and grow from step to step, up to 2e-13."""
    return {"rel": {"arcade": 2e-10, "adjoint": 1e-12}.get(case["family"], 3e-14)}


# --------------------------------------------------------------------------------------------
# The same equations in whole-grid torch operations
# --------------------------------------------------------------------------------------------

class _Axis:
    def __init__(self, d: np.ndarray, ax: int, periodic: bool, device):
        self.ax, self.n = ax, len(d)
        self.lo, self.hi = (0, len(d) - 1) if periodic else (2, len(d) - 3)
        v = torch.as_tensor(np.ascontiguousarray(d), device=device)
        self.d = v[:, None] if ax == 0 else v[None, :]
        self.h = 0.5 * self.d
        self.fden = self.h + self.roll(self.h, 1)

    def roll(self, q, k: int):
        """q of the cell k places below (k > 0) or above (k < 0)."""
        return torch.roll(q, k, self.ax)

    def face(self, q):
        """Interpolation to the face below each cell."""
        return (self.roll(q, 1) * self.h + q * self.roll(self.h, 1)) / self.fden

    def diff(self, f):
        return (self.roll(f, -1) - f) / self.d

    def deriv(self, q):
        return self.diff(self.face(q))

    def second(self, q):
        f = self.face(q)
        return (self.roll(f, -1) - 2.0 * q + f) / (self.h * self.h)

    def upwind(self, q, v):
        """Barton-limited upwind value at the face below each cell for the face velocity v."""
        h, pos = self.h, v > 0.0
        a, b = torch.where(pos, self.roll(q, 2), self.roll(q, -1)), torch.where(pos, self.roll(q, 1), q)
        g = torch.where(pos, self.roll(h, 2) + 2.0 * self.roll(h, 1), self.roll(h, -1) + 2.0 * h)
        e = torch.where(pos, self.roll(self.fden, 1), self.roll(self.fden, -1))
        d1, d2 = a + (b - a) * g / e, self.face(q)
        low = (q <= self.roll(q, 1)) == pos
        inner = torch.where(low == (d1 < d2), d2, d1)
        lim = torch.where(low == (inner < b), inner, b)
        return torch.where(v != 0.0, lim, d2)


class _Exact:
    """Mesh, boundary kinds and constants of a spec, on the device."""

    def __init__(self, spec: DomainSpec):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.spec, self.bc = spec, spec.bc
        self.x = _Axis(spec.grids["d_x"][:, 0], 0, spec.bc[0] == PERIODIC, self.dev)
        self.y = _Axis(spec.grids["d_y"][0, :], 1, spec.bc[2] == PERIODIC, self.dev)
        m = torch.zeros((spec.xdim, spec.ydim), dtype=torch.bool, device=self.dev)
        m[self.x.lo:self.x.hi + 1, self.y.lo:self.y.hi + 1] = True
        self.inside = m
        self.gm1 = spec.adiabatic_index - 1.0

    def grid(self, name: str):
        return torch.as_tensor(self.spec.grids[name], device=self.dev)

    def mask(self, q):
        return torch.where(self.inside, q, torch.zeros_like(q))


class _Mhd(_Exact):
    """u = [rho, mom_x, mom_y, mom_z, thermal_energy, bi_x, bi_y, bi_z]."""

    def __init__(self, spec: DomainSpec):
        super().__init__(spec)
        self.be = [self.grid(k) for k in ("be_x", "be_y", "be_z")]
        self.g = [self.grid(k) for k in ("grav_x", "grav_y")]
        self.m = spec.ion_mass
        n = torch.clamp(self.grid("rho") / self.m, min=spec.density_min)
        te = 2.0 * n * K_B * torch.clamp(self.grid("temp"), min=spec.temp_min) / self.gm1
        self.start = self.propagate([self.grid("rho")] + [self.grid(k) for k in ("mom_x", "mom_y", "mom_z")] + [te] +
                                    [self.grid(k) for k in ("bi_x", "bi_y", "bi_z")])

    def minimums(self, u):
        u = list(u)
        u[0] = torch.clamp(u[0] / self.m, min=self.spec.density_min) * self.m
        u[4] = torch.clamp(u[4], min=self.spec.thermal_energy_min)
        return u

    def propagate(self, u):
        u = self.minimums(u)
        if self.bc[2] == FIXED:   # lower side
            for k in (1, 2, 3):
                u[k] = torch.cat([torch.zeros_like(u[k][:, :3]), u[k][:, 3:]], 1)
        if self.bc[3] == OPEN:    # upper side, no boost and no decay
            d = self.y.d[0]
            rho, te = u[0][:, -3], u[4][:, -3]
            vx, vy = u[1][:, -3] / rho, u[2][:, -3] / rho
            bv = torch.clamp(vy, min=0.0)
            gv = (0.5 * (d[-2] + d[-3]) * bv - 0.5 * d[-2] * vy) / (0.5 * d[-3])
            ghost = {0: rho, 1: rho * vx, 2: rho * gv, 4: te}
            for k, v in ghost.items():
                u[k] = torch.cat([u[k][:, :-2], v[:, None], v[:, None]], 1)
        return self.minimums(u)

    def temp(self, rho, te):
        return torch.clamp(te * self.gm1 / (2.0 * K_B * rho / self.m), min=self.spec.temp_min)

    def step_size(self, u):
        rho, press = u[0], u[4] * self.gm1
        b2 = sum((a + b) ** 2 for a, b in zip(self.be, u[5:]))
        cs2, va2 = press * self.spec.adiabatic_index / rho, b2 / (rho * (4.0 * math.pi))
        s = cs2 + va2
        delta = torch.sqrt(torch.clamp(1.0 - 4.0 * cs2 * va2 / (s * s), min=1e-300))
        c = torch.sqrt(s * 0.5 * (1.0 + delta))
        dt = 1.0 / ((torch.abs(u[1] / rho) + c) / self.x.d + (torch.abs(u[2] / rho) + c) / self.y.d)
        dt = dt[self.inside]
        return self.spec.epsilon * dt[torch.argmin(dt.detach())]

    def rhs(self, u):
        rho, te, b, be = u[0], u[4], u[5:], self.be
        v = [m / rho for m in u[1:4]]
        press = te * self.gm1
        moved = [rho, u[1], u[2], u[3], te, b[0], be[0], b[1], be[1], b[2], be[2]]
        t = [0.0] * 11
        for ax, w in ((self.x, v[0]), (self.y, v[1])):
            vf = ax.face(w)
            t = [a + ax.diff(ax.upwind(q, vf) * vf) for a, q in zip(t, moved)]
        ddx, ddy = self.x.deriv, self.y.deriv
        four_pi = 4.0 * math.pi
        curl = (ddx(b[1]) - ddy(b[0])) / four_pi
        cz0, cz1 = ddy(b[2]), -ddx(b[2])
        bt = [p + q for p, q in zip(b, be)]
        vx, vy = [ddx(q) for q in v], [ddy(q) for q in v]
        k = [-t[0],
             -t[1] - ddx(press) + rho * self.g[0] - curl * bt[1] + bt[2] * cz1 / four_pi,
             -t[2] - ddy(press) + rho * self.g[1] + curl * bt[0] - bt[2] * cz0 / four_pi,
             -t[3] + (cz0 * bt[1] - cz1 * bt[0]) / four_pi,
             -t[4] - press * (vx[0] + vy[1])]
        k += [-t[5 + 2 * i] - t[6 + 2 * i] + bt[0] * vx[i] + bt[1] * vy[i] for i in range(3)]
        return [self.mask(q) for q in k]

    def advance(self, u, h, k):
        return self.minimums([a + h * b for a, b in zip(u, k)])

    def bhat(self, u):
        b = [p + q for p, q in zip(self.be, u[5:])]
        n = torch.sqrt(b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
        return b[0] / n, b[1] / n

    # conduction
    def saturated(self, T, rho, bx, by, dsm):
        gx, gy = self.mask(self.x.deriv(T)), self.mask(self.y.deriv(T))
        kap = torch.minimum(1e-6 * T ** 2.5, self.x.d * self.y.d * K_B * (rho / self.m) / dsm)
        f = -kap * (gx * bx + gy * by)
        fx, fy = f * bx, f * by
        sat = rho / self.m * 0.25 * (T * K_B) ** 1.5 / math.sqrt(M_ELECTRON)
        fm = torch.sqrt(fx * fx + fy * fy)
        return gx * bx + gy * by, fx, fy, fm, sat / torch.sqrt(sat * sat + fm * fm)

    def conduction(self, te, rho, bx, by, saturation, dsm):
        X, Y = self.x, self.y
        T = self.temp(rho, te)
        gx, gy = self.mask(X.deriv(T)), self.mask(Y.deriv(T))
        bdg = bx * gx + by * gy
        bxx, bxy, byx, byy = X.deriv(bx), Y.deriv(bx), X.deriv(by), Y.deriv(by)
        curl = byx - bxy
        sx = bx * X.second(T) + by * Y.deriv(gx) + gx * bxx + gy * bxy + curl * gy
        sy = bx * X.deriv(gy) + by * Y.second(T) + gx * byx + gy * byy - curl * gx
        p15, p25 = T * torch.sqrt(T), T * T * torch.sqrt(T)
        r = p25 * bdg * (bxx + byy) + bx * (2.5 * p15 * gx * bdg + p25 * sx) + by * (2.5 * p15 * gy * bdg + p25 * sy)
        r = self.mask(r * 1e-6)
        if saturation:
            _, fx, fy, fm, coef = self.saturated(T, rho, bx, by, dsm)
            coef = torch.where(self.inside & (fm != 0.0), coef, torch.ones_like(coef))
            r = self.mask(coef * r - (X.deriv(coef) * self.mask(fx) + Y.deriv(coef) * self.mask(fy)))
        return r

    def losses(self, te, rho):
        T = self.temp(rho, te)
        one = torch.ones_like(T)
        lg = torch.log10(T)
        table = ((4.97, 1.09e-31, T * T), (5.67, 8.87e-17, 1.0 / T), (6.18, 1.90e-22, one), (6.55, 3.53e-13, T ** -1.5),
                 (6.90, 3.46e-25, T ** (1.0 / 3.0)), (7.63, 5.49e-16, 1.0 / T))
        chi = 1.96e-27 * torch.sqrt(T)
        for top, c, p in reversed(table):
            chi = torch.where(lg <= top, c * p, chi)
        n = rho / self.m
        chi = n * n * chi
        chi = torch.where(T < 5e4, chi * ((T - 3e4) / 2e4), chi)
        return self.mask(torch.where(T < 3e4, torch.zeros_like(T), chi))

    def modules(self, u, h, case):
        """Conduction and radiation before the integrator; their subcycle counts from the step's start."""
        sat, rk2, dsm = case.get("saturation", False), case.get("tc_integrator") == "rk2", 1e-6
        bx, by = self.bhat(u)
        rho, te = u[0], u[4]
        with torch.no_grad():
            T, size = self.temp(rho, te), self.x.d * self.y.d
            scale = K_B / 1e-6 * (rho / self.m) * size / T ** 2.5
            if sat:
                ftg, _, _, fm, c = self.saturated(T, rho, bx, by, dsm)
                scale = torch.nan_to_num(K_B / torch.abs(c * fm / ftg) * (rho / self.m) * size, nan=1e300)
            n_tc = int(float(h) / max(0.5 * float(scale[self.inside].min()), dsm)) + 1
            loss = self.losses(te, rho)
            n_rl = int(float(h) / (0.5 * float((te / loss)[self.inside].abs().min()))) + 1 if float(loss.max()) else 0
        floor = self.spec.thermal_energy_min
        for _ in range(n_tc):
            mid = te
            if rk2:
                mid = torch.clamp(te + 0.5 * (h / n_tc) * self.conduction(te, rho, bx, by, sat, dsm), min=floor)
            te = torch.clamp(te + (h / n_tc) * self.conduction(mid, rho, bx, by, sat, dsm), min=floor)
        u = self.propagate(u[:4] + [te] + u[5:])
        te = u[4]
        for _ in range(n_rl):
            te = torch.clamp(te - (h / n_rl) * self.losses(te, u[0]), min=floor)
        return self.propagate(u[:4] + [te] + u[5:])

    def heating(self, theta):
        y = torch.as_tensor(self.spec.grids["pos_y"][0], device=self.dev)
        w = (y.max() - y.min()) / 15.0
        at = y.min() + w * torch.arange(16, device=self.dev, dtype=torch.float64)
        phi = torch.exp(-0.5 * ((y[None, :] - at[:, None]) / w) ** 2)
        return self.mask((theta @ phi)[None, :].expand(self.spec.xdim, self.spec.ydim))

    def steps(self, u, case, theta=None):
        dts = []
        for _ in range(case["steps"]):
            h = self.step_size(u)
            dts.append(h)
            if self.spec.modules:
                u = self.modules(u, h, case)
            if self.spec.integrator == RK2:
                u = self.advance(u, h, self.rhs(self.advance(u, 0.5 * h, self.rhs(u))))
            else:
                k1 = self.rhs(u)
                k2 = self.rhs(self.advance(u, 0.5 * h, k1))
                k3 = self.rhs(self.advance(u, 0.5 * h, k2))
                k4 = self.rhs(self.advance(u, h, k3))
                u = self.advance(u, h, [(a + d) / 6.0 + (b + c) / 3.0 for a, b, c, d in zip(k1, k2, k3, k4)])
            u = self.propagate(u)
            if theta is not None:
                u = self.propagate(u[:4] + [u[4] + h * self.heating(theta)] + u[5:])
        return u, torch.stack(dts)


class _TwoFluid(_Exact):
    """u in TF_EVOLVED order, without the curl terms (B and E_z stay zero)."""

    def __init__(self, spec: DomainSpec):
        super().__init__(spec)
        self.mass = (spec.ion_mass, M_ELECTRON)
        rho = [self.grid("i_rho"), self.grid("e_rho")]
        te = [r / m * K_B * self.grid(k) / self.gm1 for r, m, k in zip(rho, self.mass, ("i_temp", "e_temp"))]
        z = torch.zeros_like(rho[0])
        self.start = self.ghost(self.minimums(rho + [z] * 4 + te + [z] * 2))

    def minimums(self, u):
        u = list(u)
        for s in range(2):
            u[s] = torch.clamp(u[s] / self.mass[s], min=self.spec.density_min) * self.mass[s]
            u[6 + s] = torch.clamp(u[6 + s], min=self.spec.thermal_energy_min)
        return u

    def ghost(self, u):
        out = []
        for q in u:
            q = q.clone()
            q[:2, 2:-2], q[-2:, 2:-2] = q[2, 2:-2].clone(), q[-3, 2:-2].clone()
            q[2:-2, :2], q[2:-2, -2:] = q[2:-2, 2:3].clone(), q[2:-2, -3:-2].clone()
            out.append(q)
        return out

    def step_size(self, u):
        n, te = u[1] / M_ELECTRON, u[7] * self.gm1 / (K_B * (u[1] / M_ELECTRON))
        wpe2, vth2 = 4 * math.pi * n * E_CHARGE * E_CHARGE / M_ELECTRON, K_B * te / M_ELECTRON
        s = 0.0
        for ax, m in ((self.x, u[4]), (self.y, u[5])):
            k = 2.0 * math.pi / (2 * ax.d)
            s = s + (torch.abs(m / u[1]) + torch.sqrt(wpe2 + 3 * k * k * vth2) / k) / ax.d
        return self.spec.epsilon * (1.0 / s)[self.inside].min()

    def rhs(self, u):
        k = [None] * 10
        cur = [0.0, 0.0]
        for s in range(2):
            rho, m, te = u[s], (u[2 + 2 * s], u[3 + 2 * s]), u[6 + s]
            v = [q / rho for q in m]
            t, div = [0.0] * 4, 0.0
            for ax, w in ((self.x, v[0]), (self.y, v[1])):
                vf = ax.face(w)
                t = [a + ax.diff(ax.upwind(q, vf) * vf) for a, q in zip(t, (rho, m[0], m[1], te))]
                div = div + ax.diff(vf)
            press, q = te * self.gm1, (1.0 - 2.0 * s) * E_CHARGE * rho / self.mass[s]
            k[s] = -t[0]
            for i, ax in enumerate((self.x, self.y)):
                k[2 + 2 * s + i] = -t[1 + i] - ax.deriv(press) + q * u[8 + i]
                cur[i] = cur[i] + q * v[i]
            k[6 + s] = -t[3] - press * div
        k[8], k[9] = -4.0 * math.pi * cur[0], -4.0 * math.pi * cur[1]
        return [self.mask(q) for q in k]

    def steps(self, u, steps: int):
        dts = []
        for _ in range(steps):
            h = self.step_size(u)
            dts.append(h)
            mid = self.ghost(self.minimums([a + 0.5 * h * b for a, b in zip(u, self.rhs(u))]))
            u = self.ghost(self.minimums([a + h * b for a, b in zip(u, self.rhs(mid))]))
        return u, torch.stack(dts)


def exact(case: dict, seed: int) -> Optional[dict]:
    if case["family"] == "plasma":
        got = []
        for spec in _plasma_specs(case, seed):
            E = _TwoFluid(spec)
            got.append(E.steps(E.start, case["steps"]))
        if case["members"] == 1:
            return {"dt": got[0][1], **dict(zip(TF_EVOLVED, got[0][0]))}
        return {"dt": torch.stack([g[1] for g in got]), "members": [torch.stack(g[0]) for g in got]}
    spec = _mhd_spec(case, seed)
    E = _Mhd(spec)
    u = E.propagate(E.start)
    if case["family"] != "adjoint":
        with torch.no_grad():
            u, dts = E.steps(u, case)
        return {"dt": dts, **dict(zip(MHD_EVOLVED, u))}
    u0 = [q.detach().clone().requires_grad_(True) for q in u]
    theta = torch.as_tensor(_theta(), device=E.dev).requires_grad_(True) if case["arcade"] else None
    u, dts = E.steps(u0, case, theta)
    lam = torch.as_tensor(_loss_seed(case, spec, seed), device=E.dev)
    J = sum((a * b).sum() for a, b in zip(lam, u))
    wrt = u0 + ([theta] if theta is not None else [])
    g = torch.autograd.grad(J, wrt)
    out = {"dt": dts.detach(), "grad": dict(zip(MHD_EVOLVED, g)), **{k: q.detach() for k, q in zip(MHD_EVOLVED, u)}}
    if theta is not None:
        out["grad_theta"] = g[8]
    return out
