"""Calls whose batches run in different segment shapes on one context: a lone
query below 2e15 takes smaller segments than a batch, or the no-allocation entry
point, does.  Results are integers: tolerance 0."""
import pytest

pytestmark = pytest.mark.gpu


# the documented use of the no-allocation call: an allocating call at the largest
# x has built the tables
@pytest.mark.parametrize("x", [10 ** 9, 10 ** 10, 10 ** 11, 10 ** 12, 10 ** 15])
def test_noalloc_after_a_lone_query(x):
    import cudapix_amd as C
    with C.Context(device=0) as c:
        want = c.pi_batch([x])
        assert c.pi_batch_noalloc([x]) == want
        assert c.pi_batch_noalloc([x, x // 2]) == [want[0], c.pi(x // 2)]


@pytest.mark.parametrize("x", [10 ** 9, 10 ** 10, 10 ** 11])
def test_noalloc_after_one_solve(x):
    import cudapix_amd as C
    with C.Context(device=0) as c:
        assert [c.pi(x)] == c.pi_batch_noalloc([x])
