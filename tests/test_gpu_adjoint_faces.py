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
