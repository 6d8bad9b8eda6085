"""The one pass that forms b_hat and the modules' subcycle-count reductions, and the radiative subcycles
with the propagate that ends them, against the CPU restatement (correctly rounded powers), bit for bit:
grids of less than one 64x4 block, of whole blocks and of a column or row more; conduction alone, radiation
alone, both, both with flux saturation and the radiation's step-size guard, and two radiation modules (the
second needs a pass of its own)."""
import numpy as np
import pytest

from oracle.oracle import OracleDomain, set_pow_mode
from spruce_amd import workloads as W
from spruce_amd.gpu import GpuDomain
from spruce_amd.spec import spec_from_files
from tests.bits import same_bits
from tests.test_gpu_tc_strip import VARS, describe

pytestmark = pytest.mark.gpu

RL = ("radiative_losses", [("cutoff_ramp", "2e4"), ("cutoff_temp", "3e4"), ("epsilon", "0.1")])
RL_PREVENT = ("radiative_losses", RL[1] + [("prevent_subcycling", "true"), ("time_integrator", "rk2")])


def _tc(sat):
    return ("thermal_conduction", [("flux_saturation", sat), ("epsilon", "0.5"), ("dt_subcycle_min", "1e-4")])


@pytest.fixture
def cr_oracle():
    set_pow_mode(1)
    yield
    set_pow_mode(0)


@pytest.mark.parametrize("nx,ny,mods", [
    (5, 5, [_tc("false"), RL]), (8, 64, [_tc("false")]), (9, 65, [RL]), (13, 63, [RL_PREVENT, _tc("true")]),
    (17, 130, [_tc("true"), RL]), (11, 70, [RL, RL_PREVENT])])
def test_modules_match_cr_restatement(nx, ny, mods, cr_oracle):
    print("step pre", nx, ny, [m[0] for m in mods], flush=True)
    st = W.arcade_state(nx, ny, dx=5e6, dy0=5e6, stretch=1.01, t_corona=2e6)
    st.grids["temp"] = st.grids["temp"] * (1.0 + 0.01 * (2 * W.uniform(nx * ny, (nx, ny)) - 1))
    cfg = W.base_config("ideal_mhd", ("periodic", "periodic", "fixed", "open"), "rk2", epsilon=0.2, max_iterations=4,
                        density_min=1.0, temp_min=1e4, thermal_energy_min=1e-8, modules=mods)
    spec = spec_from_files(cfg, st)
    g, o = GpuDomain(spec), OracleDomain(spec)
    try:
        for s in range(3):
            dg, sg = g.step(1, subcycles=True)
            do = o.step(1)
            assert list(sg[0]) == o.subcycles() and same_bits(dg, do), (s, sg[0], o.subcycles(), dg, do)
        for v in VARS:
            a, b = g.grid(v), o.grid(v)
            assert same_bits(a, b), "%s: %s" % (v, describe(np.asarray(a), np.asarray(b)))
    finally:
        g.close()
        o.close()
