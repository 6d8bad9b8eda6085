"""GPU parity: the HIP path through the C ABI against the golden vectors of the compiled reference
and against the CPU restatement, bit for bit (integer-exact comparison of the FP64 bit patterns),
with identical dt sequences."""
import numpy as np
import pytest

from golden_util import golden_names, load_golden
from oracle.oracle import OracleDomain
from spruce_amd import workloads as W
from spruce_amd.gpu import GpuDomain, arith_probe
from spruce_amd.spec import spec_from_files
from tests.bits import same_bits

pytestmark = pytest.mark.gpu

MHD_VARS = ["rho", "temp", "mom_x", "mom_y", "mom_z", "bi_x", "bi_y", "bi_z", "n", "thermal_energy", "press",
            "v_x", "v_y", "v_z", "kinetic_energy", "b_x", "b_y", "b_z", "b_mag", "b_hat_x", "b_hat_y", "b_hat_z", "dt"]


def describe(a, b):
    d = np.abs(a - b) / np.maximum(np.abs(b), 1e-300)
    k = np.unravel_index(np.nanargmax(d), d.shape)
    return "max rel diff %.3e at %s (%r vs %r), %d cells differ" % (d[k], k, a[k], b[k], int(np.sum(a != b)))


def test_device_division_and_sqrt_are_ieee():
    rng = np.random.default_rng(1)
    n = 1 << 20
    a = np.ldexp(rng.uniform(1, 2, n), rng.integers(-300, 300, n)) * rng.choice([-1, 1], n)
    b = np.ldexp(rng.uniform(1, 2, n), rng.integers(-200, 200, n))
    a[:1000] = 0.0
    d, s, q = arith_probe(a, b)
    assert same_bits(d, a / b)
    assert same_bits(q, a / b)
    # exponents on both sides of the thresholds where the corrected-reciprocal quotient hands over to
    # the IEEE division (|a| near 2^+-700, |a/b| near 2^+-850)
    a2 = np.ldexp(rng.uniform(1, 2, n), rng.integers(-720, 720, n)) * rng.choice([-1, 1], n)
    b2 = np.ldexp(rng.uniform(1, 2, n), rng.integers(-170, 170, n))
    _, _, q2 = arith_probe(a2, b2)
    assert same_bits(q2, a2 / b2)
    pos = np.abs(a)
    _, s2, _ = arith_probe(pos, b)
    assert same_bits(s2, np.sqrt(pos))


# the solar cases go through libm pow in the reference and are compared within tolerance in
# test_gpu_modules.py; every other case is bit-identical
@pytest.mark.parametrize("case", [c for c in golden_names() if c.startswith(("mhd_", "tf_", "e2_", "cons_"))])
def test_gpu_matches_reference_golden(case):
    g = load_golden(case)
    dom = GpuDomain(g.spec())
    try:
        for name, ref in g.frame(0).items():
            got = dom.grid(name)
            assert same_bits(got, ref), "%s setup %s: %s" % (case, name, describe(got, ref))
        step = 0
        for k in g.frames[1:]:
            dts = dom.step(k - step)
            assert same_bits(dts, g.dt_steps[step:k]), "%s dt sequence %s vs %s" % (case, dts, g.dt_steps[step:k])
            step = k
            for name, ref in g.frame(k).items():
                got = dom.grid(name)
                assert same_bits(got, ref), "%s frame %d %s: %s" % (case, k, name, describe(got, ref))
    finally:
        dom.close()


def _random_case(nx, ny, seed, bc, integ, **kw):
    from tests.golden.cases import random_mhd_state
    st = random_mhd_state(nx, ny, seed, stretch=kw.pop("stretch", False))
    cfg = W.base_config("ideal_mhd", bc, integ, epsilon=0.2, density_min=1.0, temp_min=1.0,
                        thermal_energy_min=1e-12, **kw)
    return spec_from_files(cfg, st)


BIG = [
    ("periodic_rk2", ("periodic",) * 4, "rk2", {}),
    ("open_rk4", ("open",) * 4, "rk4", dict(open_boundary_strength=0.5, open_boundary_decay_base=0.6, stretch=True)),
    ("fixed_euler", ("fixed",) * 4, "euler", {}),
    ("reflect_rk2", ("reflect",) * 4, "rk2", dict(stretch=True)),
    ("ucnp_rk4", ("open_ucnp",) * 4, "rk4", {}),
    ("mixed_rk2", ("periodic", "periodic", "fixed", "open"), "rk2", dict(open_boundary_strength=0.3)),
    # no ghost fill between the final stage, which forms the next step size, and its use
    ("periodic_euler", ("periodic",) * 4, "euler", dict(stretch=True)),
    ("periodic_rk4", ("periodic",) * 4, "rk4", {}),
]


# strips of the default height (1 row on this grid), of several rows with remainders, and one over the whole grid
KERNELS = [("strip", None), ("strip", 4), ("strip", 12), ("cell", None), ("strip", 136)]


@pytest.mark.parametrize("kernel,rows", KERNELS, ids=["strip", "strip4", "strip12", "cell", "strip136"])
@pytest.mark.parametrize("name,bc,integ,kw", BIG, ids=[b[0] for b in BIG])
def test_gpu_matches_oracle_multi_block(name, bc, integ, kw, kernel, rows):
    spec = _random_case(133, 197, 7, bc, integ, **dict(kw))
    ora = OracleDomain(spec)
    gpu = GpuDomain(spec, options={"stage_kernel": kernel, **({"strip_rows": rows} if rows else {})})
    try:
        rg, ro = gpu.rhs(), ora.rhs()
        assert same_bits(rg, ro), "rhs: " + describe(rg, ro)
        for _ in range(3):
            dg, do = gpu.step(4), ora.step(4)
            assert same_bits(dg, do), "dt %s vs %s" % (dg, do)
        for v in MHD_VARS:
            a, b = gpu.grid(v), ora.grid(v)
            assert same_bits(a, b), "%s %s: %s" % (name, v, describe(a, b))
        assert gpu.time == ora.time
    finally:
        gpu.close()
        ora.close()


@pytest.mark.parametrize("kernel", ["auto", "cell", "tile"])
def test_periodic_workload_full_size_matches_oracle(kernel):
    """"tile" is a name that is still accepted: it runs strips."""
    st = W.periodic_wave_state(256, 256, seed=0)
    spec = spec_from_files(W.periodic_wave_config(steps=1000), st)
    ora = OracleDomain(spec)
    gpu = GpuDomain(spec, options={"stage_kernel": kernel})
    try:
        dg, do = gpu.step(5), ora.step(5)
        assert same_bits(dg, do)
        for v in ("rho", "mom_x", "mom_y", "thermal_energy", "bi_x", "bi_y", "n", "temp", "dt"):
            assert same_bits(gpu.grid(v), ora.grid(v)), v
    finally:
        gpu.close()
        ora.close()


def test_translation_equivariance_at_2048():
    """A periodic uniform mesh has no preferred cell: shifting the input shifts every output bit for bit."""
    st = W.periodic_wave_state(2048, 2048, seed=5)
    cfg = W.periodic_wave_config(steps=10)
    sx, sy = 389, 1021
    st2 = W.periodic_wave_state(2048, 2048, seed=5)
    for k in ("rho", "temp", "mom_x", "mom_y", "mom_z", "bi_x", "bi_y", "bi_z", "grav_x", "grav_y"):
        st2.grids[k] = np.roll(st.grids[k], (sx, sy), axis=(0, 1))
    a = GpuDomain(spec_from_files(cfg, st))
    b = GpuDomain(spec_from_files(cfg, st2))
    try:
        da, db = a.step(3), b.step(3)
        assert same_bits(da, db)
        for v in ("rho", "mom_x", "thermal_energy", "bi_y"):
            assert same_bits(np.roll(a.grid(v), (sx, sy), axis=(0, 1)), b.grid(v)), v
        assert np.all(da > 0)
    finally:
        a.close()
        b.close()
