"""The operand ranges of spruce_amd/csrc/range.hpp keep every untested division of the stencils exact.

Each value is bounded as (lo, g, hi): 0, or of magnitude 2**lo .. 2**hi, and a multiple of 2**g.  A sum
of multiples of 2**g is one, so it is 0 or at least 2**g; a double of magnitude at least 2**lo is a
multiple of 2**(lo - 52).  The chains below are the kernels' own: whatever they divide must be 0 or at
least 2**-960 (the residual b*q - a of qdiv_in is then exact), the quotient at least 2**-960 too, and
nothing may reach 2**900.  Where the divisor is data, recip_in also bounds the divisor and the quotient,
and sqrt_in its argument (range.hpp).
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


G, L, U, R, RU, RCP, Q = (CONST["RANGE_" + k] for k in "G L U R RU RCP Q".split())
H = magnitude(-G, G)                # halves, sums of halves, cell sizes, extrapolation weights
FOUR_PI = magnitude(3, 4)
GM1, GAMMA = magnitude(-60, 10), magnitude(0, 11)           # gamma - 1 is checked at set-up
M_E, K_B, E_CH, C = magnitude(-90, -89), magnitude(-53, -52), magnitude(-31, -30), magnitude(34, 35)
POW_IN = 200                        # crpow.hpp: pow_1p5_2p5_in takes 2**-200 .. 2**200


def test_constants():
    for x, v in ((FOUR_PI, 12.566370614359172), (M_E, 9.1093837e-28), (K_B, 1.380649e-16), (E_CH, 4.80320425e-10),
                 (C, 2.99792458e10)):
        assert 2.0 ** x.lo <= v <= 2.0 ** x.hi


def recip_div(x, y, quotient=None):
    """qdiv_in(x, y, recip_in(y)); quotient: its bounds where x and y are not independent."""
    assert x.lo >= -960 and x.hi <= 900 and -RCP <= y.lo and y.hi <= RCP
    lo, hi = quotient or (x.lo - y.hi, x.hi - y.lo)
    assert -Q <= lo and hi <= Q, "quotient 2**%d .. 2**%d" % (lo, hi)
    return magnitude(lo, hi)


def sqrt_in(x):
    assert -RCP <= x.lo and x.hi <= RCP
    return magnitude(x.lo // 2, -(-x.hi // 2))


def positive_sum(*v):
    """A sum of values that are not negative, the first of them positive."""
    hi = max(x.hi for x in v) + len(v) - 1
    return magnitude(v[0].lo, hi)


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
    v = recip_div(q, rho)                                 # v = mom / rho
    vf = interp(v)
    for x in (q, rho):
        diff(limited(x) * vf)                             # transport divergence
    diff(interp(q))                                       # derivative1D of pressure (times gamma-1), bi
    press = q * GM1
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
    recip_div(T * den, den, (T.lo, T.hi))                 # te (gamma - 1) = T den
    for x in (T, T * K_B):                                # T^1.5 and T^2.5, (T K_B)^1.5
        assert -POW_IN <= x.lo and x.hi <= POW_IN
    hsq = magnitude(-2 * G, 2 * G)
    f = interp(T)
    qdiv_in(f + T + f, hsq)                               # second derivative
    g = diff(f)
    diff(interp(g))                                       # derivative of the other axis's gradient
    diff(interp(b))


def test_stage_step_size():
    """dt_inverse: rho, te, mom and |b|^2 of the updated cell are tested, te is positive."""
    q, te, rho, b2 = magnitude(-L, U), magnitude(-L, U), magnitude(-R, RU), magnitude(-L, U)
    v = recip_div(q, rho)
    cs = sqrt_in(recip_div(te * GM1 * GAMMA, rho))
    va = recip_div(sqrt_in(b2), sqrt_in(rho * FOUR_PI))
    cs2, va2 = cs * cs, va * va
    s = positive_sum(cs2, va2)
    # 4 c v / (c + v)^2 is at most 1, and at least the smaller of c / v and v / c
    ratio = max(cs2.hi - va2.lo, va2.hi - cs2.lo)
    recip_div(cs2 * magnitude(2, 2) * va2, s * s, (-ratio - 1, 1))
    vfast = sqrt_in(s * magnitude(-1, -1) * magnitude(0, 1))   # 1 + delta lies in 1 .. 2
    qdiv_in(positive_sum(either(cs, vfast), va, v), H)
    assert 2 * v.lo > -1000 and 2 * v.hi < 1000           # |v| stands for sqrt(v*v)


def test_two_fluid_chains():
    """The species' transport is the stage's; mass: an ion mass checked at set-up, or the electron's."""
    q, rho, b = magnitude(-L, U), magnitude(-R, RU), magnitude(-L, U)
    v = recip_div(q, rho)
    for mass in (magnitude(-150, 40), M_E):
        num = qdiv_in(rho, mass)
        num * E_CH * v                                    # the current
        num * E_CH * qdiv_in(v * b, C)                    # the force's v x B / c
    C * diff(interp(b))                                   # the curl terms


def test_two_fluid_step_size():
    """tf_dt_inverse: the electrons' rho, te and mom of the updated cell are tested, te is positive."""
    q, te, rho = magnitude(-L, U), magnitude(-L, U), magnitude(-R, RU)
    v = recip_div(q, rho)
    k = magnitude(1 - (G - 2), 2 + (G - 2))               # pi / d, d checked at set-up
    en = qdiv_in(rho, M_E)
    etemp = recip_div(te * GM1, K_B * en)
    vth = sqrt_in(qdiv_in(K_B * etemp, M_E))
    wpe = sqrt_in(qdiv_in(FOUR_PI * en * E_CH * E_CH, M_E))
    wth = sqrt_in(k * k * magnitude(1, 2) * (vth * vth))
    w = sqrt_in(positive_sum(wpe * wpe, wth * wth))
    qdiv_in(positive_sum(recip_div(w, k), v), H)


def test_ranges_cover_ordinary_states():
    """Far wider than any state of the workloads: density 1e-45..1e12 g/cm3, other values 1e-51..1e45."""
    assert 2.0 ** -R < 1e-40 and 2.0 ** RU > 1e10
    assert 2.0 ** -L < 1e-50 and 2.0 ** U > 1e40
    assert 2.0 ** (2 - G) < 1e-12 and 2.0 ** (G - 2) > 1e12
