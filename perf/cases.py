"""The workloads this library is timed on, through its Python interface.

A case is a dict of plain values; `prepare` makes its queries from a seed and
keeps the context (and server) a program would keep from call to call, `run`
makes one pass, `work` states the arithmetic the answer cannot do without and
`exact` recomputes small answers without the library.

A pass costs what the query costs: inputs and results are a few bytes, the
resident tables stay with the context, and the time is sieving and lookups.
"""
import json
import math
import random

import numpy as np

import cudapix_amd as C

TERMS = ("pi", "ordinary", "trivial", "easy", "hard", "p2")


def listed():
    return [
        # one small query, the latency of a call: a command line or a script
        # asking for a single value
        {"name": "pi_1e9", "kind": "pi", "x": 10 ** 9},
        # the smaller of the two single-query sizes the benchmark reports
        {"name": "pi_1e12", "kind": "pi", "x": 10 ** 12},
        # the larger one, the size single queries are tuned at
        {"name": "pi_1e16", "kind": "pi", "x": 10 ** 16},
        # a research-size query of 64 bits
        {"name": "pi_1e18", "kind": "pi", "x": 10 ** 18},
        # x above 2^64: the 128-bit path, the longest pass here
        {"name": "pi_2e19", "kind": "pi", "x": 2 * 10 ** 19},
        # every table rebuilt for the call: a one-shot solve, and the plain
        # rate the batched one is compared with
        {"name": "pi_1e13_fresh", "kind": "pi", "x": 10 ** 13, "fresh": True},
        # the terms one by one with a y of the caller's choice, as a program
        # written against the term functions calls them
        {"name": "terms_1e14", "kind": "terms", "x": 10 ** 14, "alpha": 2.5},
        # the benchmark's batch: 512 queries log-uniform in [1e9, 1e15], two
        # batches in flight, at the benchmark's tuning
        {"name": "batch_512", "kind": "batch", "n": 512, "lo": 9.0, "hi": 15.0, "batches": 2, "tuned": True},
        # an odd-sized batch of larger queries with default options, every
        # term of every query returned
        {"name": "batch_47_terms", "kind": "batch", "n": 47, "lo": 11.0, "hi": 16.0, "batches": 1,
         "terms": True},
        # a burst of requests to the server in each of its modes
        {"name": "served_batches_300", "kind": "served", "n": 300, "lo": 9.0, "hi": 15.0,
         "mode": "batches", "tuned": True},
        {"name": "served_stream_100", "kind": "served", "n": 100, "lo": 9.0, "hi": 14.0, "mode": "stream"},
        # primes of a window far above the resident table
        {"name": "count_1e14", "kind": "count", "lo": 10 ** 14, "n": 1 << 32},
    ]


def draw(rng):
    kind = rng.choice(["pi", "pi", "pi", "fresh", "terms", "batch", "batch", "served", "served", "count"])
    if kind == "pi":
        return {"kind": "pi", "x": int(10 ** rng.uniform(9, 19.2))}
    if kind == "fresh":
        return {"kind": "pi", "x": int(10 ** rng.uniform(10, 15)), "fresh": True}
    if kind == "terms":
        return {"kind": "terms", "x": int(10 ** rng.uniform(11, 15)), "alpha": rng.uniform(1.2, 5.0)}
    if kind == "batch":
        hi = rng.uniform(11, 15.5)
        return {"kind": "batch", "n": int(2 ** rng.uniform(2, 9)), "lo": rng.uniform(5, hi), "hi": hi,
                "batches": rng.choice([1, 2, 3]), "tuned": rng.random() < 0.5, "terms": rng.random() < 0.5}
    if kind == "served":
        hi = rng.uniform(11, 15)
        return {"kind": "served", "n": int(2 ** rng.uniform(3, 8.5)), "lo": rng.uniform(6, hi), "hi": hi,
                "mode": rng.choice(["batches", "stream"]), "tuned": rng.random() < 0.5}
    return {"kind": "count", "lo": int(10 ** rng.uniform(10, 15)), "n": int(10 ** rng.uniform(6, 9.8))}


# The context (and server) of the case in use: a program makes one and solves
# everything with it, so states of one case share it.
_kept = {"key": None, "ctx": None, "server": None}


def _handles(case):
    key = json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)
    if _kept["key"] != key:
        if _kept["server"] is not None:
            _kept["server"].close()
        if _kept["ctx"] is not None:
            _kept["ctx"].close()
        _kept.update(key=None, ctx=None, server=None)
        ctx = C.Context(device=0, fresh_tables=bool(case.get("fresh")))
        _kept["ctx"] = ctx
        if case.get("tuned"):
            ctx.set_tuning(512, 32, 0.3, 8)
        if case["kind"] == "served":
            mode = C.SERVER_BATCHES if case["mode"] == "batches" else C.SERVER_STREAM
            _kept["server"] = C.Server(ctx, max_batch=512, mode=mode, max_x=int(10 ** case["hi"]) + 1)
        _kept["key"] = key
    return _kept["ctx"], _kept["server"]


def _inputs(case, seed):
    """The integers of a state: x within 2 % above the case's, or the list of queries."""
    rng = random.Random("%s %d" % (case["kind"], seed))
    if case["kind"] in ("pi", "terms"):
        return case["x"] + rng.randrange(case["x"] // 50)
    if case["kind"] == "count":
        return case["lo"] + rng.randrange(case["lo"] // 50)
    return [[int(10 ** rng.uniform(case["lo"], case["hi"])) for _ in range(case["n"])]
            for _ in range(case.get("batches", 1))]


def _icbrt(x):
    r = int(round(x ** (1 / 3)))
    while r ** 3 > x:
        r -= 1
    while (r + 1) ** 3 <= x:
        r += 1
    return r


def _y(case, x):
    return int(case["alpha"] * _icbrt(x))


def prepare(case, seed):
    ctx, server = _handles(case)
    return {"case": case, "ctx": ctx, "server": server, "in": _inputs(case, seed)}


def run(state):
    case, ctx, what = state["case"], state["ctx"], state["in"]
    if case["kind"] == "pi":
        return ctx.pi(what)
    if case["kind"] == "terms":
        x, y = what, _y(case, what)
        return {"P2": ctx.P2(x, y), "S0": ctx.Ordinary(x, y), "S1": ctx.S2_trivial(x, y), "S3": ctx.S3(x, y),
                "V": ctx.V(x, y)}
    if case["kind"] == "count":
        return ctx.countPrimes(what, what + case["n"])
    if case["kind"] == "served":
        tickets = [state["server"].submit(x) for x in what[0]]
        state["server"].drain()
        got = {r["ticket"]: r["pi"] for r in state["server"].poll(len(tickets) + 16)}
        return np.array([got[t] for t in tickets], dtype=np.int64)
    if case.get("terms"):
        return [np.array([[t[k] for k in TERMS] for t in ctx.pi_batch(xs, terms=True)], dtype=np.int64)
                for xs in what]
    return [np.array(r, dtype=np.int64) for r in ctx.pi_batches(what)]


def _pi_ops(x):
    """x^(2/3) / ln^2 x: operations of the combinatorial method."""
    return x ** (2 / 3) / math.log(x) ** 2


def work(case):
    if case["kind"] in ("pi", "terms"):
        return {"bytes": 32, "flops": _pi_ops(case["x"])}
    if case["kind"] == "count":
        # a sieve marks every integer once for each of its small primes
        return {"bytes": 24, "flops": case["n"] * math.log(math.log(case["lo"] + case["n"]))}
    n = case["n"] * case.get("batches", 1)
    grid = [10 ** (case["lo"] + (case["hi"] - case["lo"]) * (k + 0.5) / 64) for k in range(64)]
    return {"bytes": 32 * n, "flops": n * sum(map(_pi_ops, grid)) / 64}


def _pi_exact(x):
    """pi(x) by sieving the values floor(x / k), prime by prime."""
    r = math.isqrt(x)
    low = np.arange(r + 1, dtype=np.int64) - 1           # counts at 0 .. r
    high = np.zeros(r + 1, dtype=np.int64)               # counts at x // k
    high[1:] = x // np.arange(1, r + 1, dtype=np.int64) - 1
    for p in range(2, r + 1):
        if low[p] == low[p - 1]:
            continue
        before, p2 = low[p - 1], p * p
        if p2 > x:
            break
        top = min(r, x // p2)
        k = np.arange(1, top + 1, dtype=np.int64)
        inside = min(top, r // p)
        high[1:inside + 1] -= high[p * k[:inside]] - before
        rest = k[inside:]
        high[inside + 1:top + 1] -= low[x // (p * rest)] - before
        if p2 <= r:
            v = np.arange(p2, r + 1, dtype=np.int64)
            low[p2:] -= low[v // p] - before
    return int(high[1])


def exact(case, seed):
    # every answer is a whole number; the larger ones take a sieve of hours
    if case["kind"] == "pi" and case["x"] <= 2 * 10 ** 12:
        return _pi_exact(_inputs(case, seed))
    return None
