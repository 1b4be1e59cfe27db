"""The segment sieve's bitmap of the integers coprime to 30, at its edges:
every wheel (the hard leaves of the stages below the sieve's own wheel come in
closed form), intervals that end on and beside a segment or a wave's bits, and
groups of every number of member slots.  Everything is an integer, so every
comparison is for equality."""
import pytest

pytestmark = pytest.mark.gpu

TERMS = ("ordinary", "trivial", "easy", "hard", "p2", "pi")
SEG = 30 * 256 * 32 * 32 // 8          # integers of a segment of 256 threads x 32 words
WAVE = 30 * 64 * 32 * 32 // 8


def _same(t, ref, what):
    for k in TERMS:
        assert t[k] == ref[k], (what, k, t[k], ref[k])


# x^(1/4) on both sides of 11, 13, 17, 19, 23 and 29: wheels of 5 to 8 primes, and the
# first sieved stages above them
@pytest.mark.parametrize("x", [16384, 28560, 28561, 83520, 83521, 130320, 130321, 279840, 279841, 707281,
                               5 * 10 ** 6 + 1, 10 ** 9 + 7])
def test_every_wheel(ctx, oracle, x):
    for c in range(1, 9):
        for alpha in (1.0, 2.3):
            y = oracle.choose_y(x, alpha)
            _same(ctx.pi(x, y=y, c=c, terms=True), oracle.pi_dr(x, y, c), (x, c, y))
            assert ctx.S3(x, y, c=c) == oracle.pi_dr(x, y, c)["hard"], (x, c, y)


# z = floor(x / y) on the last integer of a segment or wave, the first of the next, and around
@pytest.mark.parametrize("end", [WAVE, SEG, 2 * SEG, 2 * SEG + 3 * WAVE])
@pytest.mark.parametrize("d", [-30, -1, 0, 1, 30])
def test_interval_ends(ctx, oracle, end, d):
    y = 2003
    x = y * (end + d) + 5
    _same(ctx.pi(x, y=y, terms=True), oracle.pi_dr(x, y, 6), (x, y))


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 31, 32, 33, 65])
def test_group_sizes(ctx, oracle, n):
    xs = [3 * 10 ** 9 + 1234567 * k for k in range(n)]
    xs[0] = 10 ** 9 + 9                   # a member whose interval ends early
    got = ctx.pi_batch(xs, terms=True)
    for k in sorted({0, 1 % n, n // 2, n - 1}):
        _same(got[k], oracle.pi_dr(xs[k], got[k]["y"], int(got[k]["c"])), (n, k))
    assert [t["pi"] for t in got] == [ctx.pi(x) for x in xs]


# every shape, with x large enough for stages on both sides of each way of crossing off
@pytest.mark.parametrize("shape", [(64, 32), (64, 128), (256, 64), (256, 128), (512, 64)])
def test_shapes_term_by_term(ctx, shape):
    import cudapix_amd as C
    xs = [10 ** 13 + 7 * k for k in range(9)]
    want = ctx.pi_batch(xs, terms=True)
    with C.Context(device=0, seg_threads=shape[0], seg_kwords=shape[1]) as c:
        for t, u in zip(c.pi_batch(xs, terms=True), want):
            _same(t, u, shape)
        _same(c.pi(10 ** 16, terms=True), ctx.pi(10 ** 16, terms=True), shape)


# the hard carry takes a stage's rows in 32 runs, four rows of a run at a time: numbers of
# segments on both sides of one row a run, four rows a run and their remainders (y on both
# sides of the least it can be, so that the numbers of stages differ)
@pytest.mark.parametrize("nseg", [1, 2, 4, 31, 32, 33, 63, 65, 127, 128, 129, 133])
@pytest.mark.parametrize("extra", [2, 301])
def test_carry_runs(ctx, oracle, nseg, extra):
    z = SEG * nseg - 7
    y = max(int(z ** 0.5) + extra, 100)
    x = y * z + 3
    _same(ctx.pi(x, y=y, terms=True), oracle.pi_dr(x, y, 6), (x, y))


# the P2 primes of a segment: counted by its first replica or shared by all of them, on both
# sides of the rule, with y near and far from sqrt(x) and groups of several queries
@pytest.mark.parametrize("x", [10 ** 9, 3 * 10 ** 10 + 1, 10 ** 11, 7 * 10 ** 11 + 9, 10 ** 12, 10 ** 13 + 37])
@pytest.mark.parametrize("alpha", [1.0, 4.0, 17.0])
def test_p2_shared(ctx, oracle, x, alpha):
    y = oracle.choose_y(x, alpha)
    ref = oracle.pi_dr(x, y, 6)
    _same(ctx.pi(x, y=y, terms=True), ref, (x, y))
    assert ctx.P2(x, y) == ref["p2"], (x, y)


# the prime sieve of a P2 range by waves: 64 primes a wave at a time (all stage counts from
# none, and the last prime below and at the square root of the segment's end)
@pytest.mark.parametrize("x", [SEG, SEG + 1, 10 ** 7 + 19, 1400 ** 3, 1409 ** 3 - 1, 10 ** 10 - 33])
def test_p2_wave_primes(ctx, oracle, x):
    for alpha in (1.0, 2.0, 6.0):
        y = oracle.choose_y(x, alpha)
        _same(ctx.pi(x, y=y, c=4, terms=True), oracle.pi_dr(x, y, 4), (x, y))
