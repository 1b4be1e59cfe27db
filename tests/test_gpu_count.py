"""Prime counts by the segmented sieve, at the edges of its ways of crossing off
(primes below 1024, 16384 and 2^18 and above), of its words of 120 integers and of
its segments.  Counts, so every comparison is for equality."""
import pytest

pytestmark = pytest.mark.gpu

SEG = 40960 * 120


@pytest.fixture()
def fresh():
    import cudapix_amd as C
    with C.Context(device=0) as c:          # no resident table: every count comes from the sieve
        yield c


@pytest.mark.parametrize("lo,hi", [(0, 1), (0, 2), (2, 3), (0, 3), (1, 20), (19, 20), (20, 24), (0, 121), (7, 120),
                                   (119, 121), (120, 240), (1021, 1033), (16381, 16412), (262139, 262152),
                                   (0, SEG - 1), (0, SEG), (0, SEG + 1), (0, 3 * SEG + 7), (SEG - 1, SEG + 2)])
def test_small_windows(fresh, oracle, lo, hi):
    assert fresh.countPrimes(lo, hi) == oracle.count_primes(lo, hi)


# p^2 around each bound, and windows of one integer to several segments
@pytest.mark.parametrize("root", [23, 1021, 1031, 16381, 16411, 262139, 262147, 10 ** 6 + 3])
@pytest.mark.parametrize("n", [1, 119, 1000, 2 * SEG + 61])
def test_windows_at_squares(fresh, oracle, root, n):
    for lo in (root * root - n, root * root - n // 2, root * root):
        lo = max(lo, 0)
        assert fresh.countPrimes(lo, lo + n) == oracle.count_primes(lo, lo + n), (lo, n)


# the pi table's segments (32768 integers for a table of up to 2^28, 131072 above): counts from
# the table beside and across their ends and at its end, against the sieve of a context without it
@pytest.mark.parametrize("x", [10 ** 10, 10 ** 15, 7 * 10 ** 16, 8 * 10 ** 16])
def test_table_segments(oracle, x):
    import cudapix_amd as C
    top = int(x ** 0.5)
    ends = [k * 32768 for k in (1, 2, 3, 4, 8)] + [top // 131072 * 131072, top // 32768 * 32768]
    with C.Context(device=0) as c, C.Context(device=0) as d:
        c.pi(x)
        for e in ends:
            if e > top:
                continue
            for lo, hi in ((e - 1000, e), (e - 1, e + 2), (max(e - 131072, 0), min(e + 32768, top))):
                assert c.countPrimes(lo, hi) == d.countPrimes(lo, hi), (x, lo, hi)
        assert c.countPrimes(0, top) == d.countPrimes(0, top), x
