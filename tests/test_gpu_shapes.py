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


def _lone_shape(c, x=10 ** 12):
    st = c.pi_batch([x], stats=True)[1]
    return st["seg_threads"], st["seg_kwords"]


# a tuner that fails (an x it cannot plan, an allocation that fails) leaves the
# context as it found it: its shape and factors, the lone query's own shape, and
# a later tune that runs
@pytest.mark.parametrize("how", ["range", "alloc 2", "alloc 9"])
def test_failed_tune_leaves_the_context(how):
    import cudapix_amd as C
    xs = [10 ** 11, 10 ** 11 + 99, 10 ** 12]
    with C.Context(device=0) as c:
        before, lone = c.tuning(), _lone_shape(c)
        assert lone != (before["seg_threads"], before["seg_kwords"])
        for call in (c.autotune, lambda v: c.pi_batch(v, tune=True)):
            try:
                if how != "range":
                    C.debug_fail_alloc(int(how.split()[1]))
                with pytest.raises(C.CpxError):
                    call(xs + [10 ** 30] if how == "range" else [100 * x for x in xs])
            finally:
                C.debug_fail_alloc(0)
            assert c.tuning() == before and _lone_shape(c) == lone
        want = [c.pi(x) for x in xs]
        assert c.pi_batch(xs, tune=True) == want
        t = c.tuning()
        assert _lone_shape(c) == (t["seg_threads"], t["seg_kwords"])


# lone queries between batches, with shapes of their own (below 2e15) and the
# context's: every result as alone, and no graph captured again on the way
def test_lone_queries_between_batches():
    import cudapix_amd as C
    many = [10 ** 11 + 12345 * k for k in range(20)]
    lone = [10 ** 9, 10 ** 12 + 1, 3 * 10 ** 15, 10 ** 13 + 7]
    with C.Context(device=0) as c:
        want, alone = [c.pi(x) for x in many], [c.pi(x) for x in lone]
        for x in lone:                           # tables and arena at their largest
            c.pi_batch([x])
        c.pi_batch(many)
        n = c.graph_captures()
        for _ in range(3):
            for x, v in zip(lone, alone):
                assert c.pi_batch([x]) == [v]
                assert c.pi_batch(many) == want
        assert c.graph_captures() == n


# a batch-mode server whose budget holds a lone request's state in the context's shape
# only, and one that holds a few requests of a burst at a time
@pytest.mark.parametrize("xs,budget,least", [([10 ** 15], 3600000, 1), ([10 ** 12 + 3 ** k for k in range(24)], 2500000, 2)])
def test_batch_server_within_its_budget(ctx, xs, budget, least):
    import cudapix_amd as C
    with C.Context(device=0) as c:
        srv = C.Server(c, hbm_budget=budget, mode=C.SERVER_BATCHES)
        tickets = [srv.submit(x) for x in xs]
        srv.drain()
        res = {r["ticket"]: r for r in srv.poll(100)}
        st = srv.stats()
        srv.close()
    assert [(res[t]["status"], res[t]["pi"]) for t in tickets] == [(0, ctx.pi(x)) for x in xs]
    assert st["max_inflight_bytes"] <= budget and st["batches"] >= least and st["rejected"] == 0


# a wave of the shape with the longest waves crosses off more than 2^16 integers a stage if
# the caller's wheel leaves it the stages of 3 and 5 (the sieve's own wheel does not)
@pytest.mark.parametrize("c", [1, 2, 4])
@pytest.mark.parametrize("x", [10 ** 9 + 7, 10715741739, 26496490190])
def test_small_wheels_in_the_longest_wave(oracle, x, c):
    import cudapix_amd as C
    with C.Context(device=0, seg_threads=64, seg_kwords=128) as k:
        t = k.pi(x, c=c, terms=True)
        ref = oracle.pi_dr(x, t["y"], int(t["c"]))
        assert [t[n] for n in ("hard", "p2", "pi")] == [ref[n] for n in ("hard", "p2", "pi")]
