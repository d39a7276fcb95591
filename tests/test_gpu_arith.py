"""The in-range FP64 operations of the kernels (dvp, dvx, sqx, recip_rho, CellQuot, by_const, quot6; fvg_device.hpp and
fvg_kernels_impl.hpp) on the device against the plain division and square root there and the IEEE operations of the
host, bit for bit, over the ranges their comments state: random significands and exponents, ends of binades, quotients
and roots next to a representable value and next to the midpoint of two, the ends of the ranges, zeros of both signs and,
where they are allowed, infinities and NaN. The device's own division is not the IEEE one for a few quotients within
2^-53 ulp of a midpoint whose divisor is just below a power of two; the operations agree with it there too."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libarith_check.so")
DVP, DVX, SQX, RECIP_RHO, CELL_QUOT, CELL_H2, BY_CONST, QUOT6, DIV, SQRT = range(10)
N = 1 << 20


def device(form, a, b=None):
    assert os.path.exists(LIB), "tests/libarith_check.so is not built: run __graft_entry__.build()"
    lib, D = C.CDLL(LIB), C.POINTER(C.c_double)
    a = np.ascontiguousarray(a, dtype=np.float64)
    b = np.ones_like(a) if b is None else np.ascontiguousarray(b, dtype=np.float64)
    out, bad = np.empty_like(a), np.empty(a.size, dtype=np.int32)
    rc = lib.arith_check(form, a.ctypes.data_as(D), b.ctypes.data_as(D), C.c_longlong(a.size), out.ctypes.data_as(D),
                         bad.ctypes.data_as(C.POINTER(C.c_int)))
    assert rc == 0, rc
    return out, bad != 0


def differ(got, want):
    """Indices whose bits differ (NaN equals NaN)."""
    return np.flatnonzero((got.view(np.uint64) != want.view(np.uint64)) & ~(np.isnan(got) & np.isnan(want)))


def check(form, a, b, want, use=None, plain=None):
    """form(a, b) has the bits of want, and of the device's own operation plain."""
    got, bad = device(form, a, b)
    bits = differ(got, want)
    if plain is not None:
        bits = np.union1d(bits, differ(got, device(plain, a, b)[0]))
    if use is not None:
        bits = bits[use(bad)[bits]]
    assert bits.size == 0, [(float(a[k]).hex(), float(b[k]).hex(), float(got[k]).hex(), float(want[k]).hex()) for k in bits[:5]]


def significands(rng, n):
    """In [1, 2): random, and within a few thousand ulp of either end of the binade."""
    s = rng.integers(0, 1 << 52, n, dtype=np.uint64)
    kind = rng.integers(0, 4, n)
    near = rng.integers(0, 4096, n, dtype=np.uint64)
    s = np.where(kind == 1, near, np.where(kind == 2, np.uint64((1 << 52) - 1) - near, s))
    return (s | np.uint64(1023 << 52)).view(np.float64)


def values(rng, n, lo, hi):
    """Positive, from 2^lo to below 2^hi."""
    return np.ldexp(significands(rng, n), rng.integers(lo, hi, n))


def quotients(rng, n, elo, ehi, qlo, qhi, alo):
    """Pairs (a, b): b > 0 in 2^elo .. 2^ehi, a / b in 2^qlo .. 2^qhi, |a| at least 2^alo."""
    b = values(rng, n, elo, ehi)
    e = np.frexp(b)[1] - 1
    lo, hi = np.maximum(qlo, alo - e + 1), np.minimum(qhi, 1022 - e)
    q = np.ldexp(significands(rng, n), (lo + rng.random(n) * np.maximum(hi - lo, 1)).astype(int))
    a = q * b
    kind = rng.integers(0, 4, n)
    a = np.where(kind == 1, np.nextafter(a, 0.0), np.where(kind == 2, np.nextafter(a, np.inf), a))
    half = q * b + 0.5 * np.spacing(q) * b   # next to a midpoint, as far as the product's rounding allows
    a = np.where(kind == 3, half, a)
    ok = np.isfinite(a) & (a >= 2.0 ** alo)
    a, b = a[ok], b[ok]
    return a * rng.choice([-1.0, 1.0], a.size), b


def midpoints(rng, n):
    """Integer significands a, b whose quotient lies within a few 2^-54 ulp of the midpoint of two doubles: 2^k a =
    (2 Q + 1) b + m for an odd m, solved for Q modulo 2^k."""
    out = []
    while len(out) < n:
        b = int(rng.integers(1 << 52, 1 << 53)) | 1
        if len(out) % 3 == 0:
            b = (1 << 53) - 1 - 2 * int(rng.integers(0, 1 << 12))
        for k in (53, 54):
            for m in range(-7, 8, 2):
                t = -m * pow(b, -1, 1 << k) % (1 << k)
                a, rest = divmod(t * b + m, 1 << k)
                if t & 1 and (1 << 53) <= t < (1 << 54) and rest == 0 and (1 << 52) <= a < (1 << 53):
                    out.append((a, b))
    return np.array(out, dtype=np.float64).T


def divided(a, b):
    """a / b by the device; all but a few quotients next to a midpoint are the IEEE ones."""
    q, _ = device(DIV, a, b)
    assert differ(q, a / b).size < 1e-3 * q.size
    return q


ZEROS = np.array([0.0, -0.0])
SPECIAL = np.array([0.0, -0.0, np.inf, -np.inf, np.nan])


@pytest.mark.parametrize("form", [DVP, DVX])
def test_quotients(form):
    rng = np.random.default_rng(1 + form)
    for args in ((-60, 60, -60, 60, -969), (-1000, 1000, -1000, 1000, -969)):
        a, b = quotients(rng, N, *args)
        if form == DVP:   # negative divisors too, for a that is not zero (van Leer's limiter)
            b = b * rng.choice([-1.0, 1.0], b.size)
        check(form, a, b, a / b, plain=DIV)
    a, b = midpoints(rng, 20000)
    a, b = np.append(a, float.fromhex("0x1.6666666666663p+52")), np.append(b, float.fromhex("0x1.ffffffffffffbp+52"))
    for ea, eb in ((0, 0), (-900, 20), (300, -300), (500, 400)):
        x, y = np.ldexp(a, ea), np.ldexp(b, eb)
        check(form, x, y, divided(x, y))
    b = values(rng, 4096, -1000, 1000)
    for z in ZEROS:
        check(form, np.full(b.size, z), b, z / b, plain=DIV)


def test_quotients_of_special_values():
    with np.errstate(all="ignore"):
        x = np.concatenate([SPECIAL, [1.0, -1.0, 2.0 ** -969, 2.0 ** 900]])
        a, b = (v.ravel() for v in np.meshgrid(x, x))
        check(DVX, a, b, a / b, plain=DIV)


def test_roots():
    rng = np.random.default_rng(5)
    x = [values(rng, N, -767, 1023), values(rng, N, -60, 60)]
    r = values(rng, N, -300, 300)   # next to squares, and next to squares of midpoints
    sq = r * r
    mid = (r + 0.5 * np.spacing(r)) * r + 0.5 * np.spacing(r) * r
    x += [sq, np.nextafter(sq, 0.0), np.nextafter(sq, np.inf), mid, np.nextafter(mid, 0.0), np.nextafter(mid, np.inf)]
    x += [SPECIAL, np.array([2.0 ** -767, -1.0, np.finfo(float).max])]
    x = np.concatenate(x)
    with np.errstate(all="ignore"):
        check(SQX, x, np.ones_like(x), np.sqrt(x), plain=SQRT)


def test_reciprocal_density():
    rng = np.random.default_rng(6)
    x = np.concatenate([values(rng, N, -33, 1023), values(rng, N, -33, 8), [1e-10, 2.0 ** 1000, np.nextafter(2.0 ** 1000, np.inf),
                                                                        np.nextafter(2.0 ** 1000, 0.0), np.finfo(float).max, np.inf, np.nan]])
    check(RECIP_RHO, x, np.ones_like(x), 1.0 / x)


@pytest.mark.parametrize("form", [CELL_QUOT, CELL_H2])
def test_quotients_of_a_cell(form):
    """Whatever the cell holds: a quotient that CellQuot lets pass is the plain one."""
    rng = np.random.default_rng(7 + form)
    sign = rng.choice([-1.0, 1.0], N)
    with np.errstate(all="ignore"):
        for lo, hi in ((-510, -490), (190, 210), (-60, 60), (-1022, 1023)):
            a = values(rng, N, lo, hi) * sign
            b = values(rng, N, -33, 210) if form == CELL_QUOT else values(rng, N, -100, 101)
            check(form, a, b, a / b, lambda bad: ~bad)
        a = np.concatenate([SPECIAL, [2.0 ** 200, -2.0 ** 200, 2.0 ** -500, -2.0 ** -500]])
        x, y = (v.ravel() for v in np.meshgrid(a, [1e-10, 1.0, 3.0, 2.0 ** 100]))
        check(form, x, y, x / y, lambda bad: ~bad)
        ok = np.isin(x, ZEROS) | (np.abs(x) == 2.0 ** 200) | (np.abs(x) == 2.0 ** -500)
        assert np.array_equal(device(form, x, y)[1], ~ok)
    if form == CELL_QUOT:
        assert device(form, np.ones(3), np.array([np.nextafter(2.0 ** 200, np.inf), np.inf, np.nan]))[1].all()
    a, b = quotients(rng, N, -33 if form == CELL_QUOT else -100, 100, -60, 60, -500)
    check(form, a, b, a / b, lambda bad: ~bad)
    a, b = midpoints(rng, 20000)
    check(form, a, b, divided(a, b) if form == CELL_QUOT else a / b, lambda bad: np.ones_like(bad))


def test_quotients_by_constants():
    rng = np.random.default_rng(11)
    a, b = quotients(rng, N, -100, 101, -500, 500, -600)
    check(BY_CONST, a, b, a / b)
    a, b = midpoints(rng, 20000)
    check(BY_CONST, a, b, a / b)
    a, _ = quotients(rng, N, -2, 3, -950, 900, -960)
    a = np.concatenate([a, 6.0 * values(rng, N, -950, 900), ZEROS, [2.0 ** -960, 2.0 ** 905]])
    check(QUOT6, a, a, a / 6.0)
