"""Groups of more than eight queries, which only batches of much work form: every
term of every member against the same query solved alone (integers, tolerance 0),
at numbers of queries on both sides of 8 and 32 members."""
import pytest

pytestmark = pytest.mark.gpu

TERMS = ("ordinary", "trivial", "easy", "hard", "p2", "pi")


@pytest.fixture(scope="module")
def alone(ctx):
    xs = [3 * 10 ** 15 + 123456789 * k for k in range(64)] + [10 ** 12]
    return xs, [ctx.pi(x, terms=True) for x in xs]


@pytest.mark.parametrize("n", [9, 31, 32, 33, 64])
def test_large_members(ctx, alone, n):
    xs, want = alone
    for t, u in zip(ctx.pi_batch(xs[:n], terms=True), want):
        assert [t[k] for k in TERMS] == [u[k] for k in TERMS]


# a member whose interval ends in the first segments of the others'
def test_short_member(ctx, alone):
    xs, want = alone
    got = ctx.pi_batch([xs[-1]] + xs[:31], terms=True)
    for t, u in zip(got, [want[-1]] + want[:31]):
        assert [t[k] for k in TERMS] == [u[k] for k in TERMS]


# P2 primes of a group's segments, counted by one replica or shared by all: batches of
# a few queries (eight or more take P2 from lookups), every term against the oracle
@pytest.mark.parametrize("xs", [[10 ** 9 + 7, 10 ** 9 + 8], [10 ** 11, 3 * 10 ** 11 + 1, 7 * 10 ** 11 + 9],
                                [10 ** 12 + k for k in range(7)], [10 ** 10, 10 ** 12, 10 ** 13 + 37],
                                [5 * 10 ** 12 + 9 * k for k in range(4)]])
def test_p2_of_a_group(ctx, oracle, xs):
    for t, x in zip(ctx.pi_batch(xs, terms=True, p2_table=2), xs):
        ref = oracle.pi_dr(x, t["y"], int(t["c"]))
        for k in TERMS:
            assert t[k] == ref[k], (x, k, t[k], ref[k])
