"""Correctly rounded cos/pow used by the kernels, pinned against 70-digit
decimal arithmetic, and the rate at which glibc's libm (the reference's)
differs from correct rounding."""
from decimal import Decimal, getcontext

import numpy as np
import pytest

import oracle_ctypes as O

getcontext().prec = 70
PI = Decimal("3.14159265358979323846264338327950288419716939937510582097494459230781640628620899863")


def dcos(x):
    x = Decimal(x)
    k = (x / (2 * PI)).to_integral_value()
    y = x - k * 2 * PI
    s = Decimal(1)
    t = Decimal(1)
    n = 0
    y2 = y * y
    while True:
        n += 2
        t = -t * y2 / (n * (n - 1))
        if abs(t) < Decimal("1e-75"):
            break
        s += t
    return s


def test_pow_cr_correctly_rounded():
    rng = np.random.default_rng(5)
    xs = np.concatenate([10 ** rng.uniform(-6, 4, 4000), rng.uniform(0.5, 2, 2000),
                         np.array([1e-310, 5e-324, 1e300, 0.999999999999, 1.0000000001, 2.0, 0.5])])
    cr = O.pow_batch(xs, -0.2, O.LIBM_CR)
    for x, c in zip(xs, cr):
        assert float((Decimal(float(x)).ln() * Decimal(-0.2)).exp()) == c, x


def test_pow_special_values():
    x = np.array([0.0, np.inf, 1.0, -1.0, np.nan])
    r = O.pow_batch(x, -0.2, O.LIBM_CR)
    g = O.pow_batch(x, -0.2, O.LIBM_GLIBC)
    assert r[0] == np.inf and r[1] == 0.0 and r[2] == 1.0
    assert np.isnan(r[3]) and np.isnan(r[4])
    assert np.array_equal(r[:3], g[:3])


def test_cos_cr_correctly_rounded():
    rng = np.random.default_rng(6)
    xs = np.concatenate([rng.uniform(-4, 4, 1500), rng.uniform(-3000, 3000, 1500), rng.uniform(-1e7, 1e7, 500),
                         10 ** rng.uniform(-10, 0, 500),
                         np.array([1e-30, 0.0, np.pi / 2, np.pi, 355.0, 51996.5, 1e-8])])
    cc = O.cos_batch(xs, O.LIBM_CR)
    for x, c in zip(xs, cc):
        assert float(dcos(float(x))) == c, x


def test_glibc_rounding_difference_rates():
    """glibc 2.35 is not correctly rounded in a small fraction of calls; this is
    the only arithmetic difference between the kernels and the reference."""
    rng = np.random.default_rng(7)
    x = 10 ** rng.uniform(-4, 2, 400000)
    rp = np.mean(O.pow_batch(x, -0.2, O.LIBM_CR) != O.pow_batch(x, -0.2, O.LIBM_GLIBC))
    x = rng.uniform(-3000, 3000, 400000)
    rc = np.mean(O.cos_batch(x, O.LIBM_CR) != O.cos_batch(x, O.LIBM_GLIBC))
    assert rp < 3e-3 and rc < 5e-3
    print("pow(x,-0.2) glibc != CR: %.2e; cos glibc != CR: %.2e" % (rp, rc))


def test_cos_quick_phase_agrees_with_accurate_phase():
    """The quick phase returns a value only where its rounding test decides it; every such value equals
    the accurate phase's (2e6 arguments here; 1e9 checked the same way during development)."""
    rng = np.random.default_rng(5)
    n = 400000
    k = np.floor(rng.uniform(0, 1e5, n))
    x = np.concatenate([rng.uniform(-10, 10, n), rng.uniform(-1e6, 1e6, n), rng.uniform(-1.3e7, 1.3e7, n),
                        k * (np.pi / 2) + rng.uniform(-5e-7, 5e-7, n), np.ldexp(rng.uniform(0, 1, n), -rng.integers(0, 30, n))])
    q, dec, a = O.cos_phases(x)
    assert dec.mean() > 0.9
    assert np.array_equal(q[dec].view(np.uint64), a[dec].view(np.uint64))


@pytest.mark.parametrize("sine", [False, True])
def test_cos_turn_phase_agrees_with_accurate_phase(sine):
    """The quick phase over the whole-turn table: every value it decides equals the accurate phase's, near
    table points, halfway between them and near the zeros and extrema too, and it leaves few arguments
    undecided; tiny, huge, infinite and NaN arguments are left to the other phases or are right."""
    rng = np.random.default_rng(17)
    n = 200000
    step = np.pi / 512
    x = np.concatenate([rng.uniform(-10, 10, n), rng.uniform(-1e6, 1e6, n), rng.uniform(-1.3e7, 1.3e7, n),
                        np.floor(rng.uniform(-1e6, 1e6, n)) * step + rng.uniform(-1e-9, 1e-9, n),
                        (np.floor(rng.uniform(-1e4, 1e4, n)) + 0.5) * step + rng.uniform(-1e-12, 1e-12, n),
                        np.floor(rng.uniform(0, 1e5, n)) * (np.pi / 2) + rng.uniform(-5e-7, 5e-7, n)])
    q, dec, a = O.cos_turn_phases(x, sine)
    assert dec[:3 * n].mean() > 0.999
    assert np.array_equal(q[dec].view(np.uint64), a[dec].view(np.uint64))
    x = np.array([0.0, -0.0, 1e-300, -1e-12, 2.0 ** 30, -1e300, np.inf, -np.inf, np.nan])
    q, dec, a = O.cos_turn_phases(x, sine)
    assert np.array_equal(q[dec].view(np.uint64), a[dec].view(np.uint64))
    assert not dec[4:].any()


def test_sincos_joint_evaluation():
    rng = np.random.default_rng(23)
    x = np.concatenate([rng.uniform(-4, 4, 100000), rng.uniform(-1e7, 1e7, 100000), np.linspace(-7, 7, 20001),
                        np.array([0.0, -0.0, 1e-300, 2.0 ** 30, 1e300, np.inf, -np.inf, np.nan])])
    s, c = O.sincos_cr(x)
    for got, sine in ((s, True), (c, False)):
        want = O.cos_turn_phases(x, sine)[2]
        assert ((got.view(np.uint64) == want.view(np.uint64)) | (np.isnan(got) & np.isnan(want))).all()


@pytest.mark.parametrize("y", [-0.2, 1 / 3., -1.0, 0.9])
def test_pow_quick_phase_agrees_with_double_double(y):
    """Every value that the quick phase decides equals the double-double one (7e7 arguments checked the same way
    during development); zero, subnormal, negative, infinite and NaN arguments are left to it."""
    rng = np.random.default_rng(29)
    n = 200000
    x = np.concatenate([np.exp(rng.uniform(-10, 10, n)), np.exp(rng.uniform(-600, 600, n)), 1 + rng.uniform(-1e-3, 1e-3, n),
                        np.ldexp(1 + np.arange(4096) / 4096., rng.integers(-40, 40, 4096)), np.array([1.0, 2.0, 0.5])])
    q, dec, a = O.pow_phases(x, y)
    assert dec.mean() > 0.99
    assert np.array_equal(q[dec].view(np.uint64), a[dec].view(np.uint64))
    assert not O.pow_phases(np.array([0.0, -0.0, 5e-324, 1e-310, -1.0, np.inf, -np.inf, np.nan]), y)[1].any()


def test_philox_known_answers():
    """Philox4x32-10 known-answer vectors (Salmon et al., SC'11, the Random123 distribution)."""
    assert O.philox4x32_10([0, 0, 0, 0], [0, 0]) == [0x6627e8d5, 0xe169c58d, 0xbc57ac4c, 0x9b00dbd8]
    assert O.philox4x32_10([0xffffffff] * 4, [0xffffffff] * 2) == [0x408f276d, 0x41c83b0e, 0xa20bc7c6, 0x6d5451fd]
    assert O.philox4x32_10([0x243f6a88, 0x85a308d3, 0x13198a2e, 0x03707344], [0xa4093822, 0x299f31d0]) == \
        [0xd16cfe09, 0x94fdcceb, 0x5001e420, 0x24126ea1]


def test_sin_correctly_rounded_and_log():
    """sin via the cos reduction with the quadrant shifted: equal to 70-digit decimal arithmetic
    rounded once; the double-double log rounded once equals the correctly rounded log on the same
    samples (a hard case for log would need 2^-104 more accuracy; none occurs here)."""
    from decimal import Decimal, getcontext
    import math
    getcontext().prec = 70
    rng = np.random.default_rng(8)
    x = np.concatenate([rng.uniform(-10, 10, 1500), rng.uniform(-1e6, 1e6, 500), np.ldexp(rng.uniform(-1, 1, 200), -30),
                        np.floor(rng.uniform(0, 1e4, 300)) * (np.pi / 2) + rng.uniform(-1e-7, 1e-7, 300)])
    s, _ = O.sin_log(x)
    pi = Decimal("3.141592653589793238462643383279502884197169399375105820974944592307816406")

    def dsin(v):
        v = Decimal(float(v))
        k = (v / (2 * pi)).to_integral_value()
        v = v - k * 2 * pi
        term, tot, n = v, v, 1
        while abs(term) > Decimal(10) ** -68:
            term = -term * v * v / ((2 * n) * (2 * n + 1))
            tot += term
            n += 1
        return float(tot)
    ref = np.array([dsin(v) for v in x])
    assert np.array_equal(s.view(np.uint64), ref.view(np.uint64))
    assert np.mean(s == np.sin(x)) > 0.99  # glibc agrees almost everywhere
    y = np.exp(rng.uniform(-700, 700, 3000))
    _, lg = O.sin_log(y)
    refl = np.array([float(Decimal(float(v)).ln()) for v in y])
    assert np.array_equal(lg.view(np.uint64), refl.view(np.uint64))


def _datan(x):
    """atan in decimal arithmetic: three argument halvings, then the series"""
    from decimal import Decimal
    neg = x < 0
    x = -x if neg else x
    inv = x > 1
    if inv:
        x = 1 / x
    for _ in range(3):
        x = x / (1 + (1 + x * x).sqrt())
    x2, term, total, k = x * x, x, x, 1
    while True:
        term = term * x2
        t = term / (2 * k + 1)
        if t == 0 or t.adjusted() < -80:
            break
        total = total - t if k % 2 else total + t
        k += 1
    total = 8 * total
    if inv:
        total = _PI / 2 - total
    return -total if neg else total


_PI = None


def test_exp_and_atan2_correctly_rounded():
    """exp and atan2 against 70-digit decimal arithmetic rounded once (arguments of the JF12
    field's kind: logistic and exponential profiles, azimuths and elevation angles), plus
    C99's special cases of atan2."""
    from decimal import Decimal, getcontext
    import math
    global _PI
    getcontext().prec = 70
    _PI = Decimal("3.141592653589793238462643383279502884197169399375105820974944592307816406286")
    rng = np.random.default_rng(12)
    x = np.concatenate([rng.uniform(-700, 700, 800), rng.uniform(-20, 20, 1200), rng.uniform(-1e-3, 1e-3, 200),
                        np.ldexp(rng.uniform(-1, 1, 100), -40)])
    e, _ = O.exp_atan2(x, np.ones_like(x))
    ref = np.array([float(Decimal(float(v)).exp()) for v in x])
    assert np.array_equal(e.view(np.uint64), ref.view(np.uint64))
    X = np.concatenate([rng.uniform(-30, 30, 1500), rng.normal(size=300) * 1e-6, rng.uniform(0, 1e4, 200)])
    Y = np.concatenate([rng.uniform(-30, 30, 1500), rng.normal(size=300), rng.uniform(-1e-3, 1e-3, 200)])
    _, a = O.exp_atan2(X, Y)

    def datan2(y, x):
        y, x = Decimal(float(y)), Decimal(float(x))
        if x > 0:
            return _datan(y / x)
        if x < 0:
            return _datan(y / x) + (_PI if y >= 0 else -_PI)
        return _PI / 2 if y > 0 else -_PI / 2

    ref = np.array([float(datan2(y, x)) for x, y in zip(X, Y)])
    assert np.array_equal(a.view(np.uint64), ref.view(np.uint64))
    # special cases (C99 F.9.1.4)
    sx = np.array([1.0, -1.0, 0.0, -0.0, 0.0, -0.0, np.inf, -np.inf, np.inf, -np.inf, 5.0, -5.0, 0.0])
    sy = np.array([0.0, 0.0, 0.0, 0.0, -0.0, -0.0, np.inf, np.inf, 1.0, 1.0, np.inf, -np.inf, 2.0])
    _, a = O.exp_atan2(sx, sy)
    assert np.array_equal(a.view(np.uint64), np.arctan2(sy, sx).view(np.uint64))
    assert math.isnan(O.exp_atan2(np.array([np.nan]), np.array([1.0]))[1][0])


def test_fast_sincos_and_log_within_two_ulp():
    """The fast deterministic functions of the DiffusionSDE draws: within 2 ulp of the correctly rounded
    values (70-digit decimal) on the draws' ranges (angles in [-pi, 2pi), logarithms of (0, 1]) and
    beyond (angles to +-1e5, arguments to 1e300 and subnormal)."""
    from decimal import Decimal, getcontext
    import math
    getcontext().prec = 60
    rng = np.random.default_rng(31)
    x = np.concatenate([rng.uniform(-np.pi, 2 * np.pi, 3000), rng.uniform(-1e5, 1e5, 300), [0.0, 1e-300, -0.5]])
    sn, cs, _ = O.fast_sincos_log(x)
    def ulps(a, ref):
        return np.abs(a - ref) / np.spacing(np.abs(ref))
    ref_s = np.array([float(_dsin(Decimal(float(v)))) for v in x])
    ref_c = np.array([float(_dcos(Decimal(float(v)))) for v in x])
    big = np.abs(ref_s) > 1e-300
    assert ulps(sn[big], ref_s[big]).max() <= 2 and ulps(cs, ref_c).max() <= 2
    u = np.concatenate([1.0 - rng.uniform(0, 1, 3000), np.ldexp(1.0, -rng.integers(1, 1074, 200)), rng.uniform(1, 1e300, 200),
                        [1.0, 2.0, 0.5]])
    _, _, lg = O.fast_sincos_log(u)
    ref_l = np.array([float(Decimal(float(v)).ln()) for v in u])
    nz = ref_l != 0
    assert ulps(lg[nz], ref_l[nz]).max() <= 2 and np.all(lg[~nz] == 0)


def _dsin(x):
    """sin in decimal arithmetic: reduce by 2 pi, Taylor"""
    from decimal import Decimal
    pi = Decimal("3.14159265358979323846264338327950288419716939937510582097494459")
    x = x % (2 * pi)
    term, total, k = x, x, 1
    while abs(term) > Decimal(10) ** -55:
        term = -term * x * x / ((2 * k) * (2 * k + 1))
        total += term
        k += 1
    return total


def _dcos(x):
    from decimal import Decimal
    pi = Decimal("3.14159265358979323846264338327950288419716939937510582097494459")
    return _dsin(x + pi / 2)


def test_exp_quick_phase_equals_accurate_phase():
    """exp's quick phase (double arithmetic, Ziv rounding test at 2^-66) returns the double-double
    phase's value whenever it decides (checked on 8e7 arguments when written; 2e6 here), and decides
    almost always"""
    rng = np.random.default_rng(17)
    x = np.concatenate([rng.uniform(-708, 708, 800000), rng.uniform(-30, 30, 800000), rng.uniform(-1e-3, 1e-3, 200000),
                        np.ldexp(rng.uniform(-1, 1, 200000), -rng.integers(1, 60, 200000))])
    d, q, a = O.exp_phases(x)
    assert d.mean() > 0.999
    assert np.array_equal(q[d].view(np.uint64), a[d].view(np.uint64))


def test_atan2_quick_phase_equals_accurate_phase():
    """atan2's quick phase returns the double-double phase's value whenever it decides (8e7 argument
    pairs when written; 2e6 here across quadrants, tiny ratios and near-diagonal pairs)"""
    rng = np.random.default_rng(23)
    n = 400000
    X = np.concatenate([rng.uniform(-30, 30, n), rng.normal(size=n) * 1e-6, rng.uniform(-1, 1, n),
                        np.ldexp(rng.uniform(-1, 1, n), -rng.integers(0, 200, n)), rng.uniform(1, 2, n)])
    Y = np.concatenate([rng.uniform(-30, 30, n), rng.normal(size=n), rng.uniform(-1, 1, n) * 1e-3,
                        rng.uniform(-1, 1, n), X[-n:] * (1 + rng.uniform(-1e-9, 1e-9, n))])
    d, q, a = O.atan2_phases(Y, X)
    assert d.mean() > 0.999
    assert np.array_equal(q[d].view(np.uint64), a[d].view(np.uint64))
