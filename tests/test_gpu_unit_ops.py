"""The unit entry points put_grid, ghost_fill and propagate (PlasmaDomain::updateGhostZones,
evolution.cpp:126-152; EquationSet::propagateChanges, equationset.cpp:212-220) against the CPU
restatement, bit for bit, on every boundary kind.

The live grids are overwritten with seeded values (some densities and thermal energies below their
floors, so enforceMinimums acts), then the ghost fill alone is compared (evolved variables of the
ghost cells; derived ones keep their old values), then a whole propagate (every grid, the dt grid
and the next step size), then one more step."""
import numpy as np
import pytest

from oracle.oracle import OracleDomain
from spruce_amd import workloads as W
from spruce_amd.gpu import GpuDomain, SpruceError
from spruce_amd.spec import spec_from_files
from tests.bits import same_bits

pytestmark = pytest.mark.gpu

EVOLVED = ["rho", "mom_x", "mom_y", "mom_z", "thermal_energy", "bi_x", "bi_y", "bi_z"]
DERIVED = ["n", "temp", "press", "v_x", "v_y", "b_mag", "b_hat_x", "dt"]


def describe(a, b):
    d = np.abs(a - b) / np.maximum(np.abs(b), 1e-300)
    k = np.unravel_index(np.nanargmax(d), d.shape)
    return "max rel diff %.3e at %s, %d cells differ" % (d[k], k, int(np.sum(a != b)))


SIDES = [
    ("periodic", ("periodic",) * 4, {}),
    ("open", ("open",) * 4, dict(open_boundary_strength=0.5, open_boundary_decay_base=0.6)),
    ("fixed", ("fixed",) * 4, {}),
    ("reflect", ("reflect",) * 4, {}),
    ("ucnp", ("open_ucnp",) * 4, {}),
    ("mixed", ("periodic", "periodic", "fixed", "open"), dict(open_boundary_strength=0.3)),
    ("moc", ("periodic", "periodic", "open_moc", "open_moc"), {}),
]


def _perturbed(spec, seed):
    """Seeded replacement values for the evolved grids: 40% density and energy noise around the
    current values with a few cells pushed below the floors."""
    nx, ny = spec.xdim, spec.ydim
    u = [W.uniform(seed * 16 + k, (nx, ny)) for k in range(8)]
    rho = spec.grids["rho"] * (1.0 + 0.4 * (2 * u[0] - 1))
    rho[u[1] < 0.02] = 1e-40
    return {"rho": rho,
            "mom_x": rho * 1e7 * (2 * u[2] - 1), "mom_y": rho * 1e7 * (2 * u[3] - 1),
            "mom_z": rho * 1e6 * (2 * u[4] - 1),
            "bi_x": 0.5 * (2 * u[5] - 1), "bi_y": 0.5 * (2 * u[6] - 1), "bi_z": 0.1 * (2 * u[7] - 1)}


@pytest.mark.parametrize("name,bc,kw", SIDES, ids=[s[0] for s in SIDES])
def test_ghost_fill_and_propagate_match_restatement(name, bc, kw):
    from tests.golden.cases import random_mhd_state
    st = random_mhd_state(37, 45, 91, stretch=True)
    cfg = W.base_config("ideal_mhd", bc, "rk2", epsilon=0.2, density_min=1.0, temp_min=1.0,
                        thermal_energy_min=1e-12, **kw)
    spec = spec_from_files(cfg, st)
    print("unit ops", name, flush=True)
    gpu, ora = GpuDomain(spec), OracleDomain(spec)
    try:
        new = _perturbed(spec, 5)
        te = ora.grid("thermal_energy") * (1.0 + 0.4 * (2 * W.uniform(4321, (spec.xdim, spec.ydim)) - 1))
        te[W.uniform(4322, (spec.xdim, spec.ydim)) < 0.02] = 1e-20
        new["thermal_energy"] = te
        for v, g in new.items():
            gpu.put_grid(v, g)
            ora.put_grid(v, g)
        for v in EVOLVED:
            assert same_bits(gpu.grid(v), ora.grid(v)), "put_grid %s" % v
        gpu.ghost_fill()
        ora.ghost_fill()
        for v in EVOLVED + ["n"]:
            a, b = gpu.grid(v), ora.grid(v)
            assert same_bits(a, b), "ghost_fill %s: %s" % (v, describe(a, b))
        sg, so = gpu.propagate(), ora.propagate()
        assert same_bits(sg, so), (sg, so)
        for v in EVOLVED + DERIVED:
            a, b = gpu.grid(v), ora.grid(v)
            assert same_bits(a, b), "propagate %s: %s" % (v, describe(a, b))
        dg, do = gpu.step(1), ora.step(1)
        assert same_bits(dg, do) and same_bits(dg[0], sg), (dg, do, sg)
        for v in EVOLVED:
            a, b = gpu.grid(v), ora.grid(v)
            assert same_bits(a, b), "step %s: %s" % (v, describe(a, b))
    finally:
        gpu.close()
        ora.close()


def test_put_grid_refuses_derived_variables():
    spec = spec_from_files(W.periodic_wave_config(steps=1), W.periodic_wave_state(16, 12))
    gpu = GpuDomain(spec)
    try:
        with pytest.raises(SpruceError):
            gpu.put_grid("temp", np.ones((16, 12)))
        with pytest.raises(SpruceError):
            gpu.put_grid("rho", np.ones((12, 16)).reshape(-1)[:100])
    finally:
        gpu.close()
