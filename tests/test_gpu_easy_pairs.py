"""Easy leaves counted by the smaller prime of each pair above sqrt(x/p): the
sums against the oracle where none, some and all of a query's primes p have
their q's pass sqrt(x/p), and where sqrt(x/p) is itself a prime.  Integers, so
every comparison is for equality."""
import pytest

pytestmark = pytest.mark.gpu


def _check(ctx, oracle, x, y):
    ref = oracle.pi_dr(x, y, 6)
    t = ctx.pi(x, y=y, terms=True)
    for k in ("easy", "hard", "pi"):
        assert t[k] == ref[k], (x, y, k, t[k], ref[k])
    assert ctx.V(x, y) == ref["easy"], (x, y)
    a, b = ctx.V_split(x, y)
    assert (a, b) == (oracle.V_a(x, y), oracle.V_b(x, y)), (x, y)


@pytest.mark.parametrize("x", [10 ** 6 + 3, 10 ** 8, 10 ** 10 + 19, 10 ** 12])
@pytest.mark.parametrize("alpha", [1.0, 1.6, 4.0, 11.0, 1e9])
def test_alpha_range(ctx, oracle, x, alpha):
    _check(ctx, oracle, x, min(oracle.choose_y(x, alpha), oracle.isqrt(x)))


# x / y^2 on and beside a prime of (x^(1/4), x^(1/3)], and sqrt(x/p) = s, a prime
@pytest.mark.parametrize("p,s", [(1009, 10007), (2003, 2003), (499, 9973), (3001, 104729)])
@pytest.mark.parametrize("d", [-1, 0, 1])
def test_exact_roots(ctx, oracle, p, s, d):
    x = p * s * s + d
    for y in (s - 1, s, s + 1, 2 * s + 1):
        if oracle.icbrt(x) <= y <= oracle.isqrt(x):
            _check(ctx, oracle, x, y)
