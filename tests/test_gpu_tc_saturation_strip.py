"""Flux saturation in the strip form of the conduction update against the one-thread-per-cell form, bit
for bit: column counts around the 60-column tile of the saturated march (one column into the next tile,
one short of it) and the smallest grid, strips of 1, 2 and 5 rows (the row written lags the row formed
by one), periodic and closed sides on either axis, each subcycle integrator."""
import pytest

from spruce_amd.gpu import GpuDomain
from tests.bits import same_bits
from tests.test_gpu_tc_strip import VARS, conduction_case, describe

pytestmark = pytest.mark.gpu

PER = ("periodic",) * 4
SIDES = ("fixed", "open", "reflect", "open")
MIXED = ("periodic", "periodic", "fixed", "open")


@pytest.mark.parametrize("nx,ny,bc,integ", [
    (5, 5, PER, "euler"), (7, 59, PER, "rk2"), (8, 60, SIDES, "rk4"), (9, 61, MIXED, "rk2"), (11, 121, PER, "rk4"),
    (16, 62, SIDES, "euler"), (6, 181, MIXED, "euler")])
def test_saturated_strip_matches_cell_form(nx, ny, bc, integ):
    spec = conduction_case(nx, ny, bc, integ, True, seed=nx * ny + 1)
    print("saturated strip vs cell", nx, ny, bc, integ, flush=True)

    def run(options):
        d = GpuDomain(spec, options=options)
        try:
            dts, sub = d.step(3, subcycles=True)
            return dts, sub, {v: d.grid(v) for v in VARS}
        finally:
            d.close()

    dts_ref, sub_ref, want = run({"tc_kernel": "cell"})
    for rows in (1, 2, 5):
        dts, sub, got = run({"tc_kernel": "strip", "tc_rows": rows})
        assert (sub == sub_ref).all() and same_bits(dts, dts_ref), (rows, dts, dts_ref)
        for v in VARS:
            assert same_bits(got[v], want[v]), "rows %d %s: %s" % (rows, v, describe(got[v], want[v]))
