"""The arithmetic of the production step (mqi_prod.hpp) over the ranges that it
states: the quotients and the double square root that are to be correctly
rounded against IEEE results on the host, the others bit for bit against what
the same build makes of a division, a square root and a logarithm, and against
FP64.

Bounds against FP64: 2.5 ulp for the quotient and 3 ulp for the logarithm and
the square root, the ones that OpenCL's full profile sets for the operations
they stand for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 1 << 20
SEEDS = [1, 2, 3, 4]


def _floats(rng, lo, hi, n, signed=True):
    """Floats with exponents spread over [lo, hi) and mantissas that are
    random, short, all ones and powers of two."""
    m = rng.integers(0, 1 << 23, n)
    k = rng.integers(0, 8, n)
    m = np.where(k == 0, 0, np.where(k == 1, (1 << 23) - 1, np.where(k == 2, m >> 17 << 17, m)))
    x = np.ldexp(1.0 + m * 2.0 ** -23, rng.integers(lo, hi, n))
    return (x * np.where(rng.random(n) < 0.5, -1.0, 1.0) if signed else x).astype(np.float32)


def _doubles(rng, lo, hi, n, signed=True):
    m = rng.integers(0, 1 << 52, n)
    k = rng.integers(0, 8, n)
    m = np.where(k == 0, 0, np.where(k == 1, (1 << 52) - 1, np.where(k == 2, m >> 40 << 40, m)))
    x = np.ldexp(1.0 + m * 2.0 ** -52, rng.integers(lo, hi, n))
    return x * np.where(rng.random(n) < 0.5, -1.0, 1.0) if signed else x


def _f(ctx, fn, a, b=None):
    r = ctx.math_probe(fn, a.astype(np.float64), None if b is None else b.astype(np.float64))
    return r.astype(np.float32)


def _ulps(got, want):
    return np.abs(got.astype(np.float64) - want) / np.spacing(np.abs(want).astype(np.float32)).astype(np.float64)


@pytest.mark.parametrize("seed", SEEDS)
def test_quotient(ctx, seed):
    rng = np.random.default_rng(seed)
    a, b = _floats(rng, -60, 60, N), _floats(rng, -60, 60, N)
    q = a.astype(np.float64) / b
    ok = (np.abs(q) >= 2.0 ** -60) & (np.abs(q) <= 2.0 ** 60)
    a, b, q = a[ok], b[ok], q[ok]
    got = _f(ctx, 10, a, b)
    assert np.array_equal(got.view(np.int32), _f(ctx, 16, a, b).view(np.int32))
    assert _ulps(got, q).max() <= 2.5


@pytest.mark.parametrize("seed", SEEDS)
def test_square_root(ctx, seed):
    a = np.append(_floats(np.random.default_rng(seed), -96, 60, N, signed=False), np.float32(0))
    got = _f(ctx, 11, a)
    assert np.array_equal(got.view(np.int32), _f(ctx, 17, a).view(np.int32))
    assert _ulps(got[:-1], np.sqrt(a[:-1].astype(np.float64))).max() <= 3 and got[-1] == 0


@pytest.mark.parametrize("seed", SEEDS)
def test_logarithm(ctx, seed):
    rng = np.random.default_rng(seed)
    a = np.concatenate([_floats(rng, -126, 127, N, signed=False), _floats(rng, -3, 3, N, signed=False),
                        ((rng.integers(0, 1 << 24, N) + 1) * 2.0 ** -24).astype(np.float32)])   # the uniforms
    got = _f(ctx, 12, a)
    assert np.array_equal(got.view(np.int32), _f(ctx, 18, a).view(np.int32))
    assert _ulps(got[a != 1], np.log(a[a != 1].astype(np.float64))).max() <= 3 and (got[a == 1] == 0).all()


@pytest.mark.parametrize("seed", SEEDS)
def test_rounded_quotient(ctx, seed):
    rng = np.random.default_rng(seed)
    a, b = _floats(rng, -60, 60, N), _floats(rng, -13, 13, N)
    a[:1000] = 0
    assert np.array_equal(_f(ctx, 13, a, b), a / b)


@pytest.mark.parametrize("seed", SEEDS)
def test_rounded_double_quotient(ctx, seed):
    rng = np.random.default_rng(seed)
    a, b = _doubles(rng, -200, 200, N), _doubles(rng, -200, 200, N)
    a[:1000] = 0
    assert np.array_equal(ctx.math_probe(14, a, b), a / b)
    # operands that are floats, as most of the step's are
    a, b = _floats(rng, -60, 60, N).astype(np.float64), _floats(rng, -60, 60, N).astype(np.float64)
    assert np.array_equal(ctx.math_probe(14, a, b), a / b)


@pytest.mark.parametrize("seed", SEEDS)
def test_rounded_double_square_root(ctx, seed):
    rng = np.random.default_rng(seed)
    a = _doubles(rng, -700, 700, N, signed=False)
    assert np.array_equal(ctx.math_probe(15, a), np.sqrt(a))
    a = _doubles(rng, -80, 40, N, signed=False)   # squared step lengths
    assert np.array_equal(ctx.math_probe(15, a), np.sqrt(a))
