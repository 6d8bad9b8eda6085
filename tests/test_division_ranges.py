"""The operand ranges of spruce_amd/csrc/range.hpp keep every untested division of the stencils exact.

Each value is bounded as (lo, g, hi): 0, or of magnitude 2**lo .. 2**hi, and a multiple of 2**g.  A sum
of multiples of 2**g is one, so it is 0 or at least 2**g; a double of magnitude at least 2**lo is a
multiple of 2**(lo - 52).  The chains below are the kernels' own: whatever they divide must be 0 or at
least 2**-960 (the residual b*q - a of qdiv_in is then exact), the quotient at least 2**-960 too, and
nothing may reach 2**900.
"""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CONST = dict((k, int(v)) for k, v in re.findall(r"constexpr int (RANGE_\w+) = (\d+);",
                                                open(os.path.join(ROOT, "spruce_amd/csrc/range.hpp")).read()))


class V:
    def __init__(self, lo, g, hi):
        assert hi < 900, "may overflow"
        self.lo, self.g, self.hi = lo, g, hi

    def __add__(self, o):
        g = min(self.g, o.g)
        return V(g, g, max(self.hi, o.hi) + 1)

    def __mul__(self, o):
        return magnitude(self.lo + o.lo, self.hi + o.hi)


def magnitude(lo, hi):
    return V(lo, lo - 52, hi)


def either(*v):
    return V(min(x.lo for x in v), min(x.g for x in v), max(x.hi for x in v))


def qdiv_in(x, f):
    assert x.lo >= -960 and x.lo - f.hi >= -960, "dividend 2**%d, quotient 2**%d" % (x.lo, x.lo - f.hi)
    return magnitude(x.lo - f.hi, x.hi - f.lo)


G, L, U, R, RU = (CONST["RANGE_" + k] for k in "G L U R RU".split())
H = magnitude(-G, G)                # halves, sums of halves, cell sizes, extrapolation weights
FOUR_PI = magnitude(3, 4)


def interp(x):
    return qdiv_in(x * H + x * H, magnitude(-G, G))


def limited(x):
    """The Barton-limited face value: one of the cell's neighbours, the interpolation, the extrapolation."""
    d1 = x + qdiv_in((x + x) * H, H)
    d2 = interp(x)
    return either(x, d1, d2)


def diff(x):
    return qdiv_in(x + x, H)


def test_stage_chains():
    q = magnitude(-L, U)                                  # transported value
    rho = magnitude(-R, RU)
    v = qdiv_in(q, rho)                                   # v = mom / rho
    vf = interp(v)
    for x in (q, rho):
        diff(limited(x) * vf)                             # transport divergence
    diff(interp(q))                                       # derivative1D of pressure (times gamma-1), bi
    press = q * magnitude(-60, 10)                       # gamma - 1 is checked at set-up
    diff(interp(press))
    diff(vf)
    db = diff(interp(q))
    qdiv_in(db + db, FOUR_PI)                             # curl / 4 pi
    qdiv_in(q, FOUR_PI)
    qdiv_in(db * q + db * q, FOUR_PI)                     # (curl_z x b) / 4 pi


def test_conduction_chains():
    """The conduction update: T and n tested to 2**-100 .. 2**100 and 2**-100 .. 2**150, b_hat and the
    saturation coefficient as transported values."""
    T, b = magnitude(-100, 100), magnitude(-L, U)
    den = magnitude(-100, 150) * magnitude(-52, -51)      # n * 2 K_B
    qdiv_in(T * den, den)                                 # te (gamma - 1) = T den
    hsq = magnitude(-2 * G, 2 * G)
    f = interp(T)
    qdiv_in(f + T + f, hsq)                               # second derivative
    g = diff(f)
    diff(interp(g))                                       # derivative of the other axis's gradient
    diff(interp(b))


def test_ranges_cover_ordinary_states():
    """Far wider than any state of the workloads: density 1e-45..1e12 g/cm3, other values 1e-51..1e45."""
    assert 2.0 ** -R < 1e-40 and 2.0 ** RU > 1e10
    assert 2.0 ** -L < 1e-50 and 2.0 ** U > 1e40
    assert 2.0 ** (2 - G) < 1e-12 and 2.0 ** (G - 2) > 1e12
