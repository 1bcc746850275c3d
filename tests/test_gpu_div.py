"""The sweeps' quotients, reciprocals and square roots (csrc/satt_div.h), which
leave out the compiler's scaling of operands, against numpy's: IEEE's correctly
rounded values, the same bits over the ranges that the header states, and for
zeros, infinities and NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 1 << 22
SPECIAL = [0.0, -0.0, 1.0, -1.0, 3.0, np.inf, -np.inf, np.nan]


def operands(rng, dtype, lo, hi, n):
    """Random magnitudes of 2^lo .. 2^hi and signs; half the mantissas are within
    a few units of a power of two, where roundings of quotients are closest."""
    bits = np.finfo(dtype).nmant
    m = rng.integers(0, 1 << bits, n)
    near = rng.integers(0, 64, n)
    m = np.where(rng.random(n) < 0.25, near, np.where(rng.random(n) < 1 / 3, (1 << bits) - 1 - near, m))
    x = np.ldexp((m + (1 << bits)).astype(dtype), rng.integers(lo, hi, n) - bits)
    return (x * rng.choice([-1, 1], n)).astype(dtype)


def same(got, want):
    want = want.astype(np.float64)
    assert np.array_equal(got, want, equal_nan=True)
    fine = ~np.isnan(want)
    assert np.array_equal(np.signbit(got[fine]), np.signbit(want[fine]))


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("seed", [1, 2])
def test_quotients_are_correctly_rounded(ctx, single, seed):
    rng = np.random.default_rng(seed)
    dtype, r = (np.float32, 90) if single else (np.float64, 500)
    # operands and quotient within 2^-r .. 2^r, and, in turn, at its ends
    d = operands(rng, dtype, -r, r, N)
    q = operands(rng, dtype, -r, r, N).astype(np.float64)
    e = np.clip(np.frexp(q)[1] + np.frexp(d.astype(np.float64))[1], -r + 2, r - 2)
    n = np.ldexp(np.frexp(q)[0], e).astype(dtype)
    keep = np.abs(np.frexp(n.astype(np.float64))[1] - np.frexp(d.astype(np.float64))[1]) < r
    n, d = n[keep], d[keep]
    same(ctx.div_probe(0, n.astype(np.float64), d.astype(np.float64), single), n / d)
    # quotients within a unit of a representable number
    n = (d.astype(np.float64) * q[keep]).astype(dtype) if not single else n
    ok = np.isfinite(n) & (np.abs(np.frexp(n.astype(np.float64))[1]) < r)
    n, d = np.nextafter(n, dtype(0))[ok], d[ok]
    same(ctx.div_probe(0, n.astype(np.float64), d.astype(np.float64), single), n / d)


@pytest.mark.parametrize("single", [False, True])
def test_reciprocals_and_roots_are_correctly_rounded(ctx, single):
    rng = np.random.default_rng(3)
    dtype, r = (np.float32, 124) if single else (np.float64, 1000)
    x = operands(rng, dtype, -r, r, N)
    same(ctx.div_probe(1, x.astype(np.float64), single=single), dtype(1) / x)
    a = np.abs(operands(rng, dtype, -(100 if single else 900), 127 if single else 1023, N))
    same(ctx.div_probe(2, a.astype(np.float64), single=single), np.sqrt(a))
    if single:      # every mantissa, at an even and an odd exponent
        m = np.arange(1 << 23, dtype=np.int32)
        for e in (127, 128):
            v = (m | (e << 23)).view(np.float32)
            same(ctx.div_probe(1, v.astype(np.float64), single=True), np.float32(1) / v)
            same(ctx.div_probe(2, v.astype(np.float64), single=True), np.sqrt(v))
    else:           # squares and their neighbours
        s = np.abs(operands(rng, np.float64, -450, 500, N)) ** 2
        for v in (s, np.nextafter(s, 0), np.nextafter(s, np.inf)):
            same(ctx.div_probe(2, v), np.sqrt(v))


@pytest.mark.parametrize("single", [False, True])
def test_zeros_infinities_and_nan(ctx, single):
    dtype = np.float32 if single else np.float64
    x, y = (v.ravel() for v in np.meshgrid(SPECIAL, SPECIAL))
    with np.errstate(all="ignore"):
        same(ctx.div_probe(0, x, y, single), x.astype(dtype) / y.astype(dtype))
        same(ctx.div_probe(1, x, single=single), dtype(1) / x.astype(dtype))
        same(ctx.div_probe(2, x, single=single), np.sqrt(x.astype(dtype)))
