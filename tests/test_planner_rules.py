"""CPU test: the rules the batch planner chooses by (tests/planner_rules_check.cpp,
the engine's host code with every kernel launcher stubbed, under AddressSanitizer)."""
import os
import random
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    if not os.path.exists(HIPCC) or not shutil.which("g++"):
        pytest.skip("no hipcc")
    exe = tmp_path_factory.mktemp("planner") / "planner_rules_check"
    cmd = [HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-g",
           "-Xarch_host", "-fsanitize=address", "-fno-omit-frame-pointer",
           os.path.join(ROOT, "tests", "planner_rules_check.cpp"), "-o", str(exe), "-lpthread"]
    subprocess.run(cmd, check=True, capture_output=True)
    return exe


def run(exe, lines):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=0")
    p = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True,
                       env=env, timeout=600)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-4000:]
    out = [ln.split() for ln in p.stdout.splitlines()]
    assert len(out) == len(lines), p.stdout
    return [o[1:] for o in out]


def spread(seed, n, lo, hi):
    r = random.Random(seed)
    return [int(10 ** r.uniform(lo, hi)) for _ in range(n)]


# a batch of little work waits for the chain of the block with its first
# segments, which grows with the members: groups of eight there, of 32 above
@pytest.mark.parametrize("n,lo,hi,tuning,most", [
    (64, 9, 13, "", 8), (128, 9, 13, "", 8), (512, 9, 12, "", 8), (512, 9, 13, "", 8), (64, 12, 13, "", 8),
    (128, 9, 13, "alpha=0.3 c=8", 8), (512, 9, 12, "alpha=0.3 c=8", 8), (64, 12, 13, "alpha=0.3 c=8", 8),
    (512, 9, 15, "", 32), (512, 9, 15, "alpha=0.3 c=8", 32), (64, 14, 15, "alpha=0.3 c=8", 32),
    (256, 14, 15, "", 32), (64, 9, 13, "shape=512x64", 8), (128, 9, 13, "shape=512x64", 32),
    (128, 9, 13, "shape=256x128", 32), (128, 9, 13, "shape=256x64", 8)])
def test_group_members(checker, n, lo, hi, tuning, most):
    xs = spread(n, n, lo, hi)
    sizes = list(map(int, run(checker, ["groups %s %s" % (tuning, " ".join(map(str, xs)))])[0]))
    assert sum(sizes) == n and max(sizes) == most, sizes


# a query asks for the same tables whatever shape its batch runs in: one that a
# lone query built serves the same query in a batch or without allocation
@pytest.mark.parametrize("x", [10 ** 9, 10 ** 10, 10 ** 11, 10 ** 12, 10 ** 15, 10 ** 16, 10 ** 18])
def test_needs_in_every_shape(checker, x):
    shapes = ["64x32", "64x128", "128x64", "256x32", "256x128", "512x32", "512x64"]
    r = run(checker, ["needs %d" % x, "needs %d %d" % (x, x)] + ["needs shape=%s %d" % (s, x) for s in shapes])
    assert all(v == r[0] for v in r), r


# what a batch-mode server admits a batch by covers what the batch's plan takes: lone
# queries in the shape they run in, batches of every size over the served range
@pytest.mark.parametrize("tuning", ["", "alpha=0.3 c=8", "shape=256x32", "shape=64x32", "shape=512x64 alpha=0.5"])
def test_estimate_covers_the_plan(checker, tuning):
    lists = [[int(10 ** (e / 4))] for e in range(18, 66)] + [[2 * 10 ** 15 - 1], [5], [16384]]
    for n in (2, 3, 4, 6, 8, 9, 12, 16, 24, 32, 33, 48, 64, 100, 256):
        for lo, hi in ((5, 9), (9, 10), (9, 11), (11, 12), (12, 13), (9, 13), (13, 14), (9, 14), (14, 15), (9, 15),
                       (9, 16)):
            if n * 10 ** hi <= 2 * 10 ** 17:
                lists.append(spread(n, n, lo, hi))
    for tables in (0, 1):
        lines = ["bytes tables=%d %s %s" % (tables, tuning, " ".join(map(str, xs))) for xs in lists
                 if max(xs) < 10 ** 15 or not tables]
        for ln, (need, est) in zip(lines, run(checker, lines)):
            assert int(need) <= int(est), (ln[:80], need, est)


# a lone query keeps the context's shape where the budget holds its state in that one only
def test_lone_shape_within_budget(checker):
    for x in (10 ** 12, 10 ** 13, 10 ** 14, 10 ** 15):
        free, one = (list(map(int, r)) for r in run(checker, ["bytes %d" % x, "bytes shape=512x32 %d" % x]))
        assert one[1] < free[1]
        tight = list(map(int, run(checker, ["bytes budget=%d %d" % ((free[1] + one[1]) // 2, x)])[0]))
        assert tight == one, (x, free, one, tight)


# every descriptor list of the plan, at every wheel (x^(1/4) about 11 .. 29) with every c,
# in the lone query's shape and the context's, in batches and in other shapes
def test_descriptors(checker):
    small = [5, 16384, 28560, 28561, 83520, 83521, 130320, 130321, 279840, 279841, 707281]
    lines = ["check c=%d %d" % (c, x) for c in range(1, 9) for x in small[1:] + [10 ** 9, 10 ** 13]]
    lines += ["check %d" % int(10 ** (e / 2)) for e in range(9, 35)] + ["check tables=1 %d" % 10 ** 12]
    for n, lo, hi in ((2, 5, 9), (7, 9, 13), (8, 9, 13), (33, 4, 12), (64, 9, 14), (40, 13, 15)):
        xs = " ".join(map(str, spread(n, n, lo, hi) + small[:3]))
        lines += ["check %s %s" % (t, xs) for t in ("", "alpha=0.3 c=8", "c=1", "shape=64x32", "shape=512x64")]
    run(checker, lines)


# a block of the streaming launch claims its share of the main tiles, at most four (a cohort
# that joins waits for the tiles already claimed) and one near the end
def test_streaming_claims(checker):
    lefts = [0, 1, 511, 512, 1023, 1024, 1536, 2047, 2048, 5000, 10 ** 5, 10 ** 7]
    r = [int(v[0]) for v in run(checker, ["claim %d 512" % n for n in lefts])]
    assert r == [1, 1, 1, 1, 1, 2, 3, 3, 4, 4, 4, 4]
