"""CPU test: the benchmark's byte model counts the lookups that the easy-leaf tiles make."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("x,alpha", [(10 ** 8, 1.0), (10 ** 9, 4.0), (10 ** 9, 20.0), (10 ** 10, 2.5)])
def test_easy_pairs(x, alpha):
    sys.path.insert(0, ROOT)
    import bench
    y = int(alpha * bench.iroot(x, 3))
    primes = bench.primes_upto(bench.iroot(x, 2))
    q4, c3 = bench.iroot(x, 4), bench.iroot(x, 3)
    small = [int(p) for p in primes if p <= y]
    want = sum(1 for p in small if q4 < p <= c3 for q in small if p < q and p * p * q <= x and p * q * q <= x)
    assert bench.hbm_model_bytes([{"x": x, "y": y}], primes, 1 << 19)[1]["easy_pairs"] == want
