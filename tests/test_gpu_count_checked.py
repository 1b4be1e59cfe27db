"""Prime counts against counts made outside the library: those answered from the
resident pi table, beside and across the ends of the segments it is built in, and
those of the sieve on both sides of 2^58, where it divides differently.  Counts,
so every comparison is for equality."""
import random

import pytest

pytestmark = pytest.mark.gpu


# the table's segments hold 32768 integers up to a table of 2^28 and 131072 above
# (sqrt(7e16) = 2.65e8 and sqrt(8e16) = 2.83e8 lie on both sides)
@pytest.mark.parametrize("x", [10 ** 10, 10 ** 15, 7 * 10 ** 16, 8 * 10 ** 16])
def test_counts_from_the_table(oracle, x):
    import cudapix_amd as C
    top = oracle.isqrt(x)
    rnd = random.Random(x)
    ends = [k * 32768 for k in (1, 2, 3, 4, 8)] + [rnd.randrange(1, top // 32768 + 1) * 32768 for _ in range(8)]
    ends += [rnd.randrange(1, top // 131072 + 1) * 131072 for _ in range(8)] if top > 131072 else []
    ends += [top // 131072 * 131072, top // 32768 * 32768, top]
    with C.Context(device=0) as c:
        c.pi(x)                                  # its table reaches sqrt(x)
        for e in ends:
            if not 1 <= e <= top:
                continue
            for lo, hi in ((max(e - 1000, 0), e), (e - 1, e + 1), (max(e - 131072, 0), min(e + 32768, top))):
                assert c.countPrimes(lo, hi) == oracle.count_primes(lo, hi), (x, lo, hi)
        assert c.countPrimes(0, top) == oracle.count_primes(0, top), x


def _is_prime(n):
    """Deterministic Miller-Rabin below 3.3e24 (the first 13 primes as bases)."""
    bases = (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37, 41)
    if n < 2 or any(n % p == 0 for p in bases):
        return n in bases
    d, s = n - 1, 0
    while d % 2 == 0:
        d, s = d // 2, s + 1
    for a in bases:
        v = pow(a, d, n)
        if v in (1, n - 1):
            continue
        for _ in range(s - 1):
            v = v * v % n
            if v == n - 1:
                break
        else:
            return False
    return True


@pytest.fixture(scope="module")
def own():
    import cudapix_amd as C
    with C.Context(device=0) as c:               # (it gets a prime list to 1e9)
        yield c


@pytest.mark.parametrize("lo", [2 ** 58 - 5000, 2 ** 58 - 200, 2 ** 58, 2 ** 58 + 777, 10 ** 18 - 1, 10 ** 18 + 119])
def test_windows_about_2_58(own, lo):
    for n in (1, 120, 4001):
        assert own.countPrimes(lo, lo + n) == sum(map(_is_prime, range(lo, lo + n))), (lo, n)
