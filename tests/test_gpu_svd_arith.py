"""The Jacobi SVD's short reciprocal, quotient and square root on the device,
bit for bit against IEEE results: every significand of the reciprocal and of
the root (both exponent parities), at exponents across their ranges, and
quotients that lie as close to a rounding boundary as FP32 operands allow,
with random ones."""
import numpy as np
import pytest

import mpm_amd as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    g = M.Simulation(M.default_params((16, 16, 16), 1 / 16), 1)
    yield g
    g.close()


def _significands(exponent):
    return (np.arange(1 << 23, dtype=np.uint32) | np.uint32((exponent + 127) << 23)).view(np.float32)


def _same_bits(got, ref):
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("exponent", [-100, -1, 0, 1, 60, 99])
def test_reciprocals_of_every_significand(dev, exponent):
    y = _significands(exponent)
    _same_bits(dev.debug_svd_arith("rcp", y), np.float32(1) / y)
    _same_bits(dev.debug_svd_arith("rcp", -y), np.float32(-1) / y)


@pytest.mark.parametrize("exponent", [0, 1, 2, 61, 126, 127])
def test_roots_of_every_significand(dev, exponent):
    x = _significands(exponent)
    _same_bits(dev.debug_svd_arith("sqrt", x), np.sqrt(x))


def test_roots_of_special_values(dev):
    x = np.float32([1.0, np.inf, 4.0, np.finfo(np.float32).max])
    _same_bits(dev.debug_svd_arith("sqrt", x), np.sqrt(x))
    assert np.isnan(dev.debug_svd_arith("sqrt", np.float32([np.nan]))).all()


def _near_ties(rng, n):
    """a, b whose quotient is Q - r / b in half units of its last place, with Q
    odd (a rounding boundary) and r small: Q b = r modulo 2^25."""
    b = rng.integers(1 << 22, 1 << 23, n, dtype=np.uint64) * 2 + 1
    r = rng.integers(-16, 16, n) * 2 + 1
    inv = b.copy()
    for _ in range(5):
        inv = inv * (np.uint64(2) - b * inv)  # modulo 2^64
    Q = (inv * r.astype(np.uint64)) & np.uint64((1 << 25) - 1)
    a = (Q * b - r.astype(np.uint64)) >> np.uint64(25)
    keep = (Q >= 1 << 24) & (a > 0) & (a < 1 << 24)
    return np.float32(a[keep]), np.float32(b[keep])


@pytest.mark.parametrize("kind", ["ties", "random"])
@pytest.mark.parametrize("seed", [1, 2])
def test_quotients(dev, kind, seed):
    rng = np.random.default_rng(seed)
    n = 8000000
    if kind == "ties":
        a, b = _near_ties(rng, n)
        assert a.size > n // 3
    else:
        a, b = np.float32(rng.uniform(0.5, 2.0, n)), np.float32(rng.uniform(0.5, 2.0, n))
    ea, eb = rng.integers(-70, 20, a.size), rng.integers(-70, 20, a.size)
    a = np.ldexp(a, ea).astype(np.float32) * rng.choice(np.float32([-1, 1]), a.size)
    b = np.ldexp(b, eb).astype(np.float32) * rng.choice(np.float32([-1, 1]), a.size)
    _same_bits(dev.debug_svd_arith("div", a, b), a / b)
    zero = np.float32([0.0, -0.0, 0.0, -0.0])
    b = np.float32([1, 2, 3, 0.1])  # divisors of a rotation are positive
    _same_bits(dev.debug_svd_arith("div", zero, b), zero / b)
