"""Values outside the range of the strip kernels' untested divisions take the tested ones, bit for bit.

Each case plants values out of range (range.hpp) in part of the grid, or takes the mesh or the external
field out of range, and compares every evolved grid and step size with the CPU restatement, signs of zeros
included.
"""
import numpy as np
import pytest

from oracle.oracle import OracleDomain
from spruce_amd import workloads as W
from spruce_amd.gpu import GpuDomain
from spruce_amd.spec import spec_from_files
from tests.bits import same_bits

pytestmark = pytest.mark.gpu
PLASMA = ("i_rho", "e_rho", "i_mom_x", "i_mom_y", "e_mom_x", "e_mom_y", "i_thermal_energy", "e_thermal_energy", "E_x", "E_y",
          "E_z", "bi_x", "bi_y", "bi_z")
EVOLVED = ("rho", "mom_x", "mom_y", "mom_z", "thermal_energy", "bi_x", "bi_y", "bi_z")


def wave(nx, ny, integrator, bc, d=1e7):
    st = W.periodic_wave_state(nx, ny, d=d, seed=nx)
    g = st.grids
    g["mom_z"] = 1e-3 * g["mom_y"]
    g["bi_z"] = np.full((nx, ny), 0.5)
    return st, W.base_config("ideal_mhd", bc, integrator, epsilon=0.2, density_min=1.0, temp_min=1.0,
                             thermal_energy_min=1e-12, open_boundary_strength=0.1, open_boundary_decay_base=0.9)


def plant(st, what):
    g, i, j = st.grids, st.xdim // 2, st.ydim // 2
    if what == "tiny":          # below 2^-170, and denormal
        g["mom_z"][i:, :] = 1e-60
        g["bi_z"][:, :j] = 1e-200
        g["mom_y"][i, j] = 5e-310
    elif what == "one":         # a single cell: its strips stop at it
        g["bi_x"][i, j] = -3e-58
    elif what == "large":       # above 2^150
        g["bi_y"][i, j] = 1e46
    elif what == "zeros":       # in range: both signs of zero
        for k in ("mom_z", "bi_z"):
            g[k][:] = 0.0
        g["mom_z"][i:, :] = -0.0
    elif what == "be":
        g["be_x"] = np.full((st.xdim, st.ydim), 1e-60)


def check(st, cfg, options, steps=3, names=EVOLVED):
    spec = spec_from_files(cfg, st)
    gpu, ora = GpuDomain(spec, options), OracleDomain(spec)
    try:
        a, b = gpu.step(steps), ora.step(steps)
        assert np.array_equal(a.view(np.int64), b.view(np.int64)), (a, b)
        for v in names:
            x, y = gpu.grid(v), ora.grid(v)
            assert same_bits(x, y), (v, np.argwhere((x != y) | (np.signbit(x) != np.signbit(y)))[:4])
    finally:
        gpu.close()
        ora.close()


PERIODIC, CLOSED = ("periodic",) * 4, ("fixed", "reflect", "reflect", "fixed")


@pytest.mark.parametrize("what", ["tiny", "one", "large", "zeros", "be"])
@pytest.mark.parametrize("integrator,bc", [("rk2", PERIODIC), ("rk4", CLOSED), ("euler", ("periodic", "periodic", "fixed", "open"))])
def test_planted_values(what, integrator, bc):
    st, cfg = wave(23, 124, integrator, bc)
    plant(st, what)
    check(st, cfg, {"stage_kernel": "strip", "strip_rows": 8})


@pytest.mark.parametrize("nx,ny,rows", [(5, 5, 4), (9, 59, 4), (13, 60, 8), (16, 61, 16), (33, 121, 12)])
@pytest.mark.parametrize("bc", [PERIODIC, CLOSED])
def test_tile_edges(nx, ny, rows, bc):
    if bc is CLOSED:
        nx, ny = max(nx, 7), max(ny, 7)
    st, cfg = wave(nx, ny, "rk2", bc)
    check(st, cfg, {"stage_kernel": "strip", "strip_rows": rows})
    plant(st, "tiny")
    check(st, cfg, {"stage_kernel": "strip", "strip_rows": rows})


def test_mesh_out_of_range():
    st, cfg = wave(14, 70, "rk2", PERIODIC, d=1e-15)
    check(st, cfg, {"stage_kernel": "strip", "strip_rows": 4})


@pytest.mark.parametrize("d", [1e-302, 1e300])
def test_step_size_on_a_mesh_out_of_range(d):
    """A state at rest: the speed over the cell size overflows (a step size of 0), or is almost 0."""
    st, cfg = wave(14, 70, "rk2", PERIODIC)
    for k in ("d_x", "d_y", "pos_x", "pos_y"):
        st.grids[k] = st.grids[k] * (d / 1e7)
    for k in ("rho", "temp"):
        st.grids[k][:] = st.grids[k].mean()
    for k in ("mom_x", "mom_y", "mom_z", "bi_x", "bi_y", "bi_z"):
        st.grids[k][:] = 0.0
    check(st, cfg, {"stage_kernel": "strip", "strip_rows": 4})


@pytest.mark.parametrize("sat,integ", [(False, "euler"), (True, "rk2"), (False, "rk4")])
@pytest.mark.parametrize("what", ["bhat", "mesh"])
def test_conduction_out_of_range(sat, integ, what):
    """A field direction with a component below 2^-170 in some columns, and a mesh above 2^46."""
    from oracle.oracle import set_pow_mode
    st = W.arcade_state(22, 130, stretch=1.01)
    if what == "bhat":
        st.grids["be_x"][:, 40:90] = 1e-55
    else:
        for k in ("d_x", "d_y", "pos_x", "pos_y"):
            st.grids[k] = st.grids[k] * 1e10
        st.grids["grav_y"][:] = 0.0
    cfg = W.base_config("ideal_mhd", ("periodic", "periodic", "fixed", "open"), "rk2", epsilon=0.2, density_min=1.0, temp_min=1e4,
                        thermal_energy_min=1e-8,
                        modules=[("thermal_conduction", [("flux_saturation", str(sat).lower()), ("epsilon", "0.5"),
                                                         ("dt_subcycle_min", "1e-9"),
                                                         ("time_integrator", integ)])])
    set_pow_mode(1)
    try:
        check(st, cfg, {"tc_kernel": "strip", "tc_rows": 4}, steps=2)
    finally:
        set_pow_mode(0)


def plasma_signs(nx, ny):
    """Zero momenta of both signs beside moving cells, with everything else of the momentum equation -0 where
    v_y is: whether a momentum of -0 keeps its sign is then up to the sign of the limited fluxes' difference,
    which the untested limiter does not settle (in about one such cell in 30 it has the other one)."""
    st = W.ucnp_state(nx, ny, seed=nx)
    g, rng = st.grids, np.random.default_rng(3)
    for k in ("i_rho", "e_rho", "i_temp", "e_temp"):
        g[k] = np.full((nx, ny), g[k].max())
    for k in ("E_x", "E_y", "grav_x", "grav_y"):
        g[k] = np.full((nx, ny), -0.0)
    m = 1e4 * g["i_rho"].max()
    for k in ("i_mom_x", "e_mom_x"):
        g[k] = rng.choice([0.0, -0.0, m, -m], size=(nx, ny), p=[0.2, 0.6, 0.1, 0.1])
    for k in ("i_mom_y", "e_mom_y"):
        g[k] = rng.choice([0.0, -0.0], size=(nx, ny))
    return st


@pytest.mark.parametrize("curl", [False, True])
def test_two_fluid_momenta_of_minus_zero(curl):
    st = plasma_signs(62, 121)
    cfg = W.ucnp_config(steps=4, integrator="euler", remove_curl_terms=not curl, bc=PERIODIC)
    ora = OracleDomain(spec_from_files(cfg, st))
    try:
        ora.step(1)
        x = ora.grid("i_mom_x")
        assert 1000 < np.sum((x == 0.0) & np.signbit(x)) < np.sum(np.signbit(st.grids["i_mom_x"]) & (st.grids["i_mom_x"] == 0.0))
    finally:
        ora.close()
    for options in ({"block": "64x4"}, {"block": "strip4"}, {}):
        check(st, cfg, options, steps=1, names=PLASMA)


@pytest.mark.parametrize("curl", [False, True])
@pytest.mark.parametrize("what,nx,ny,bc", [("minus_zero", 21, 62, "open_ucnp"), ("tiny", 23, 121, "open_ucnp"),
                                           ("none", 7, 59, "fixed"), ("none", 16, 120, "reflect"), ("mesh", 14, 61, "periodic")])
def test_two_fluid(curl, what, nx, ny, bc):
    """Both species' wavefronts stop together where either finds a value out of range, or a base of -0."""
    st = W.ucnp_state(nx, ny, seed=nx, v_noise=2e4, e_noise=1e-3)
    g, i = st.grids, nx // 2
    if what == "minus_zero":
        for k in ("i_mom_x", "e_mom_y"):
            g[k][i:, :] = -0.0
    elif what == "tiny":
        g["e_mom_x"][i:i + 2, :] = 1e-70
        g["i_mom_y"][:, ny // 2:] = 1e-65
    elif what == "mesh":
        for k in ("d_x", "d_y", "pos_x", "pos_y"):
            g[k] = g[k] * 1e-15
    cfg = W.ucnp_config(steps=4, integrator="rk2", remove_curl_terms=not curl, bc=(bc,) * 4)
    check(st, cfg, {"block": "strip4"}, steps=3, names=PLASMA)
    check(st, cfg, {}, steps=3, names=PLASMA)
