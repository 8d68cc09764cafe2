"""Generate crp_crmath_tables.h: double-double constant tables for the
correctly rounded cos(), sin(), exp(), atan2(), log() and pow(x, y) used by the
propagation kernels.

Every entry is computed with Python's decimal module at 90 significant digits
and split into hi (the double nearest the value) and lo (the double nearest
the remainder), so hi + lo carries about 106 bits.

Run:  python3 crpropa3_amd/csrc/gen_crmath_tables.py > crpropa3_amd/csrc/crp_crmath_tables.h
"""
from decimal import Decimal, getcontext
import math

getcontext().prec = 90

PI = Decimal(
    "3.14159265358979323846264338327950288419716939937510582097494459230781640628620899862803482534211706798214808651"
)


def dexp(x):
    return x.exp()


def dln(x):
    return x.ln()


def dsin_cos(x):
    # Taylor series; |x| <= 1 here so 60 terms are far more than enough.
    s = Decimal(0)
    c = Decimal(0)
    term = Decimal(1)
    for n in range(0, 120):
        if n > 0:
            term = term * x / n
        r = n % 4
        if r == 0:
            c += term
        elif r == 1:
            s += term
        elif r == 2:
            c -= term
        else:
            s -= term
    return s, c


def split_dd(v):
    hi = float(v)
    lo = float(v - Decimal(hi))
    return hi, lo


def chop(v, bits):
    """v rounded to `bits` significant bits (as an exact double)."""
    f = float(v)
    m, e = math.frexp(f)
    scale = Decimal(2) ** (bits - e)
    q = (v * scale).to_integral_value()
    return float(q / scale)


def fmt(x):
    return float.hex(x)


out = []
out.append("/* Generated by gen_crmath_tables.py -- do not edit by hand. */")
out.append("/* Double-double tables: value = hi + lo to ~106 bits. */")
out.append("#ifndef CRP_CRMATH_TABLES_H")
out.append("#define CRP_CRMATH_TABLES_H")
out.append("")

# log(c_j), c_j = 1 + (j + 1/2)/256, j = 0..255
out.append("/* log(1 + (j + 0.5)/256), j = 0..255, as {hi, lo} */")
out.append("CRP_TABLE double crp_log_tab[512] = {")
for j in range(256):
    c = Decimal(1) + (Decimal(j) + Decimal("0.5")) / 256
    hi, lo = split_dd(dln(c))
    out.append("  %s, %s," % (fmt(hi), fmt(lo)))
out.append("};")
out.append("")

# 1/c_j rounded to a double, and -log of that double, for the logarithm's quick phase
out.append("/* {R_j, -log R_j hi, lo}, R_j = 1/(1 + (j + 0.5)/256) rounded, j = 0..255 */")
out.append("CRP_TABLE double crp_logr_tab[768] = {")
for j in range(256):
    r = float(1 / (Decimal(1) + (Decimal(j) + Decimal("0.5")) / 256))
    hi, lo = split_dd(-dln(Decimal(r)))
    out.append("  %s, %s, %s," % (fmt(r), fmt(hi), fmt(lo)))
out.append("};")
out.append("")

# 2^(j/256), j = 0..255
out.append("/* 2^(j/256), j = 0..255, as {hi, lo} */")
out.append("CRP_TABLE double crp_exp2_tab[512] = {")
ln2 = dln(Decimal(2))
for j in range(256):
    v = dexp(ln2 * j / 256)
    hi, lo = split_dd(v)
    out.append("  %s, %s," % (fmt(hi), fmt(lo)))
out.append("};")
out.append("")

# sin(j/32), cos(j/32), j = 0..32
out.append("/* sin(j/32), cos(j/32), j = 0..32, as {sin_hi, sin_lo, cos_hi, cos_lo} */")
out.append("CRP_TABLE double crp_sincos_tab[132] = {")
for j in range(33):
    s, c = dsin_cos(Decimal(j) / 32)
    sh, sl = split_dd(s)
    ch, cl = split_dd(c)
    out.append("  %s, %s, %s, %s," % (fmt(sh), fmt(sl), fmt(ch), fmt(cl)))
out.append("};")
out.append("")

# sin(2 pi j/1024), j = 0..767: one and a half half-turns, so that entry j + 256 is cos(2 pi j/1024) for
# j = 0..511.  The quarter-turn points are exact.
out.append("/* sin(2 pi j/1024), j = 0..767, as {hi, lo} */")
out.append("CRP_TABLE double crp_turn_tab[1536] = {")
for j in range(768):
    m = j % 512  # sin(pi + a) = -sin a
    m = min(m, 512 - m)  # sin(pi - a) = sin a
    if m <= 128:
        v = dsin_cos(2 * PI * m / 1024)[0]
    else:
        v = dsin_cos(2 * PI * (256 - m) / 1024)[1]
    if j >= 512:
        v = -v
    hi, lo = split_dd(v)
    out.append("  %s, %s," % (fmt(hi), fmt(lo)))
out.append("};")
p1 = float(2 * PI / 1024)
p2 = float(2 * PI / 1024 - Decimal(p1))
p3 = float(2 * PI / 1024 - Decimal(p1) - Decimal(p2))
out.append("/* 2 pi/1024 = P1 + P2 + P3, 53 bits each; 1024/(2 pi) */")
for i, v in enumerate((p1, p2, p3)):
    out.append("#define CRP_TURN_P%d %s" % (i + 1, fmt(v)))
out.append("#define CRP_TURN_INV %s" % fmt(float(1024 / (2 * PI))))
out.append("")

# 1/n! as dd, n = 0..20
out.append("/* 1/n!, n = 0..20, as {hi, lo} */")
out.append("CRP_TABLE double crp_invfact_tab[42] = {")
f = Decimal(1)
for n in range(21):
    if n > 0:
        f *= n
    hi, lo = split_dd(Decimal(1) / f)
    out.append("  %s, %s," % (fmt(hi), fmt(lo)))
out.append("};")
out.append("")

# 1/n as dd, n = 0..16 (entry 0 unused)
out.append("/* 1/n, n = 0..16 (entry 0 is 0), as {hi, lo} */")
out.append("CRP_TABLE double crp_recip_tab[34] = {")
out.append("  0x0p+0, 0x0p+0,")
for n in range(1, 17):
    hi, lo = split_dd(Decimal(1) / n)
    out.append("  %s, %s," % (fmt(hi), fmt(lo)))
out.append("};")
out.append("")

# pi/2 in 30-bit chunks (products with |q| < 2^23 are exact) plus a full tail
pio2 = PI / 2
parts = []
rest = pio2
for i in range(4):
    p = chop(rest, 30)
    parts.append(p)
    rest = rest - Decimal(p)
t1, t2 = split_dd(rest)
out.append("/* pi/2 = P1 + P2 + P3 + P4 + P5 + P6; P1..P4 hold 30 significant bits each */")
for i, p in enumerate(parts):
    out.append("#define CRP_PIO2_%d %s" % (i + 1, fmt(p)))
out.append("#define CRP_PIO2_5 %s" % fmt(t1))
out.append("#define CRP_PIO2_6 %s" % fmt(t2))
out.append("#define CRP_TWO_OVER_PI %s" % fmt(float(2 / PI)))
out.append("")

# ln2 in chunks for e*ln2 (|e| < 2^11): 40-bit parts
parts = []
rest = ln2
for i in range(2):
    p = chop(rest, 40)
    parts.append(p)
    rest = rest - Decimal(p)
t1, t2 = split_dd(rest)
out.append("/* ln2 = L1 + L2 + L3 + L4; L1, L2 hold 40 significant bits */")
out.append("#define CRP_LN2_1 %s" % fmt(parts[0]))
out.append("#define CRP_LN2_2 %s" % fmt(parts[1]))
out.append("#define CRP_LN2_3 %s" % fmt(t1))
out.append("#define CRP_LN2_4 %s" % fmt(t2))
out.append("")

# ln2/256 in chunks for k*ln2/256 (|k| < 2^20): 32-bit parts
l256 = ln2 / 256
parts = []
rest = l256
for i in range(2):
    p = chop(rest, 32)
    parts.append(p)
    rest = rest - Decimal(p)
t1, t2 = split_dd(rest)
out.append("/* ln2/256 = M1 + M2 + M3 + M4; M1, M2 hold 32 significant bits */")
out.append("#define CRP_LN2_256_1 %s" % fmt(parts[0]))
out.append("#define CRP_LN2_256_2 %s" % fmt(parts[1]))
out.append("#define CRP_LN2_256_3 %s" % fmt(t1))
out.append("#define CRP_LN2_256_4 %s" % fmt(t2))
out.append("#define CRP_INV_LN2_256 %s" % fmt(float(256 / ln2)))
out.append("")

# 2/pi in 32-bit words for the large-argument reduction (bits 1..1536 after the binary point),
# from pi at 500 digits (Machin: pi = 16 atan(1/5) - 4 atan(1/239)), and pi/2 as a double-double
def machin_pi(digits):
    ctx = getcontext().copy()
    ctx.prec = digits + 10

    def atan_inv(n):
        x = ctx.divide(Decimal(1), Decimal(n))
        x2 = ctx.multiply(x, x)
        term, total, k = x, x, 1
        while True:
            term = ctx.multiply(term, x2)
            t = ctx.divide(term, Decimal(2 * k + 1))
            if t == 0 or t.adjusted() < -(digits + 5):
                break
            total = ctx.subtract(total, t) if k % 2 else ctx.add(total, t)
            k += 1
        return total
    return ctx.subtract(ctx.multiply(16, atan_inv(5)), ctx.multiply(4, atan_inv(239))), ctx


pi500, ctx500 = machin_pi(500)
assert str(pi500).startswith(str(PI)[:100])
frac = ctx500.divide(Decimal(2), pi500)
words = []
for i in range(48):
    frac = ctx500.multiply(frac, Decimal(4294967296))
    w = int(frac)
    words.append(w)
    frac = ctx500.subtract(frac, Decimal(w))
out.append("/* bits of 2/pi after the binary point, 32 per word, most significant first */")
out.append("CRP_TABLE uint32_t crp_two_over_pi_bits[48] = {")
for i in range(0, 48, 6):
    out.append("    " + ", ".join("0x%08xu" % w for w in words[i:i + 6]) + ",")
out.append("};")
h, l = split_dd(ctx500.divide(pi500, Decimal(2)))
out.append("#define CRP_PIO2_DD_HI %s" % fmt(h))
out.append("#define CRP_PIO2_DD_LO %s" % fmt(l))
out.append("")
h, l = split_dd(pi500)
out.append("#define CRP_PI_DD_HI %s" % fmt(h))
out.append("#define CRP_PI_DD_LO %s" % fmt(l))
out.append("")


# atan(j/64), j = 0..64, for atan2: atan(x) = 2 atan(x / (1 + sqrt(1 + x^2))) halves the argument
# (three times), then the alternating Taylor series
def datan(x):
    ctx = getcontext()
    for _ in range(3):
        x = x / (1 + (1 + x * x).sqrt())
    x2 = x * x
    term, total, k = x, x, 1
    while True:
        term = term * x2
        t = term / (2 * k + 1)
        if t == 0 or t.adjusted() < -(ctx.prec + 5):
            break
        total = total - t if k % 2 else total + t
        k += 1
    return 8 * total


assert abs(datan(Decimal(1)) * 4 - pi500) < Decimal(10) ** -85
out.append("/* atan(j/64), j = 0..64, as {hi, lo} */")
out.append("CRP_TABLE double crp_atan_tab[130] = {")
for j in range(65):
    hi, lo = split_dd(datan(Decimal(j) / 64))
    out.append("  %s, %s," % (fmt(hi), fmt(lo)))
out.append("};")
out.append("")
out.append("#endif")
print("\n".join(out))
