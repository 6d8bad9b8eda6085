"""The face scatter of the GPU adjoint at grid sizes around its launch shapes: one row of x faces per
strip and three (both in one launch with the y faces), and two launches; strips and 61-cell tiles with
remainders.  On a uniform periodic mesh a state tiled a x b times steps as a x b copies of the small one,
bit for bit, and the gradient is linear in the seed: summed over the copies it is a*b times the gradient
of the small grid (one cell only sets the step size, so copy by copy it is not).  Both are sums of the
same terms in different orders: at most 30 additions deep per step and cell and a*b terms in the sum over
the step size, so nsteps * (30 + a*b) * 2^-53 relative to the largest entry, times 10 for the growth of a
rounding error through the reverse steps."""
import numpy as np
import pytest

from spruce_amd import workloads as W
from spruce_amd.gpu import GpuDomain
from spruce_amd.spec import spec_from_files
from spruce_amd.stateio import StateFile

pytestmark = pytest.mark.gpu

NX, NY, STEPS = 16, 21, 4
FIELDS = ("rho", "temp", "mom_x", "mom_y", "mom_z", "bi_x", "bi_y", "bi_z")


def _gradient(a, b, integ):
    rng = np.random.default_rng(7)
    st = W.periodic_wave_state(NX * a, NY * b, seed=0)
    small = W.periodic_wave_state(NX, NY, seed=0)
    g = dict(st.grids)
    for v in FIELDS:
        s = small.grids[v] * (1.0 + 0.1 * rng.uniform(-1, 1, (NX, NY)))
        g[v] = np.tile(s, (a, b))
    seed = np.tile(rng.uniform(-1, 1, (8, NX, NY)) * np.array([1e15, 1e8, 1e8, 1e8, 10, 1, 1, 1])[:, None, None],
                   (1, a, b))
    cfg = W.periodic_wave_config(steps=STEPS, integrator=integ)
    d = GpuDomain(spec_from_files(cfg, StateFile(st.xdim, st.ydim, st.ion_mass, st.adiabatic_index, st.t, g,
                                                 list(st.comments))))
    try:
        out, _ = d.adjoint(STEPS, 3, np.ascontiguousarray(seed))
    finally:
        d.close()
    out = np.asarray(out).reshape(8, a, NX, b, NY)
    return out.sum(axis=(1, 3)) / (a * b)


@pytest.mark.parametrize("a,b,integ", [(1, 3, "rk2"), (7, 11, "rk2"), (16, 13, "rk2"), (17, 9, "rk4"), (40, 14, "rk2")])
def test_tiled_state_has_the_small_grids_gradient(a, b, integ):
    print("adjoint faces", a, b, integ, flush=True)
    want, got = _gradient(1, 1, integ), _gradient(a, b, integ)
    tol = 10 * STEPS * (30 + a * b) * 2.0 ** -53
    for v in range(8):
        scale = np.abs(want[v]).max()
        print(v, scale, np.abs(got[v] - want[v]).max() / max(scale, 1e-300), tol, flush=True)
        assert scale > 0.0 or np.all(got[v] == 0.0)
        assert np.abs(got[v] - want[v]).max() <= tol * scale


SCALE = {"rho": 1e-15, "temp": 1e6, "mom_x": 1e-8, "mom_y": 1e-8, "mom_z": 1e-8, "bi_x": 1.0, "bi_y": 1.0, "bi_z": 1.0}


def _closed_run(base, grids, cfg, seed=None):
    """The evolved grids after two steps, and with a seed the gradient with respect to the state grids."""
    d = GpuDomain(spec_from_files(cfg, StateFile(base.xdim, base.ydim, base.ion_mass, base.adiabatic_index, base.t, grids,
                                                 list(base.comments))))
    try:
        if seed is not None:
            return d.adjoint_state(d.adjoint(2, 2, seed)[0])
        d.step(2)
        return np.array([d.grid(v) for v in ("rho", "mom_x", "mom_y", "mom_z", "thermal_energy", "bi_x", "bi_y", "bi_z")])
    finally:
        d.close()


@pytest.mark.parametrize("nx,ny,bc", [
    (13, 61, ("fixed", "reflect", "reflect", "fixed")), (13, 62, ("open_ucnp",) * 4), (12, 123, ("reflect", "fixed", "fixed", "open_ucnp")),
    (300, 123, ("fixed", "reflect", "reflect", "fixed")), (683, 181, ("reflect", "fixed", "open_ucnp", "reflect"))])
def test_closed_sides_at_the_edges_of_tiles(nx, ny, bc):
    """Column by column and row by row against central differences: the state is moved in one column (or row)
    next to a side or to the edge of a 61-cell tile of y faces (or in the first strips of x faces), so that a
    lost or doubled face contribution there is the whole of the difference.  Differences at two intervals
    that disagree by more than 1e-5 have crossed a switch of the limiter and are left out (few do); the others
    hold the gradient to the same 1e-5."""
    from tests.golden.cases import random_mhd_state
    base = random_mhd_state(nx, ny, nx + ny, stretch=True)
    cfg = W.base_config("ideal_mhd", bc, "rk2", epsilon=0.2, density_min=1.0, temp_min=1.0, thermal_energy_min=1e-12)
    rng = np.random.default_rng(5)
    w = rng.uniform(-1, 1, (8, nx, ny)) * np.array([1e15, 1e8, 1e8, 1e8, 10, 1, 1, 1])[:, None, None]
    g = _closed_run(base, dict(base.grids), cfg, w)
    columns = sorted({j for e in [2, ny - 3] + list(range(61, ny, 61)) for j in range(e - 2, e + 3) if 0 <= j < ny})
    rows = [0, 1, 2, 3, 4, 5, nx - 6, nx - 4, nx - 3, nx - 2, nx - 1]
    checked, worst = 0, 0.0
    for axis, k in [(1, j) for j in columns] + [(0, i) for i in rows]:
        at = np.zeros((nx, ny))
        other = rng.choice(nx if axis else ny, size=min(12, nx), replace=False)
        at[(other, k) if axis else (k, other)] = 1.0
        dirs = {v: rng.uniform(-1, 1, (nx, ny)) * s * at for v, s in SCALE.items()}
        ad = sum(float(np.sum(g[q] * dirs[v])) for q, v in enumerate(SCALE))
        fd = []
        for eps in (1e-6, 1e-7):
            out = [_closed_run(base, {v: x + sign * eps * dirs[v] if v in dirs else x for v, x in base.grids.items()}, cfg)
                   for sign in (1, -1)]
            fd.append(float(np.sum(w * (out[0] - out[1]))) / (2 * eps))
        rel = abs(ad - fd[0]) / (abs(ad) + abs(fd[0])) if ad or fd[0] else 0.0
        smooth = abs(fd[0] - fd[1]) <= 1e-5 * abs(fd[0])
        print("column" if axis else "row", k, ad, fd, "%.2e" % rel, "" if smooth else "(switch crossed)", flush=True)
        if smooth:
            checked += 1
            worst = max(worst, rel)
    assert checked >= 0.7 * (len(columns) + len(rows))
    assert worst < 1e-5
