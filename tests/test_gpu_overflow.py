"""Worklists that overflow, on the kernels of the default algorithm: marked, re-run,
reported.  What a run's smaller default worklists cannot hold is run again with larger
ones, once and not on every call.  Against the oracle."""
import numpy as np
import pytest

import oracle
from ngap_amd import Engine, NgapError
from ngap_amd.groups import make_group
from tests.test_zz_no_alloc import run_noalloc

pytestmark = pytest.mark.gpu


@pytest.fixture
def engine():
    # an engine of its own: one that a run overflowed on stays with larger worklists
    with Engine(0) as e:
        yield e


def fan(n, prefix=b"abc"):
    """After `prefix`, n states match a 'y' together, and then one reports a 'z':
    n items in one wave's queue."""
    k = len(prefix)
    return make_group(k + n + 1, [(i, i + 1) for i in range(k - 1)] +
                      [(k - 1, k + i) for i in range(n)] + [(k + i, k + n) for i in range(n)],
                      [[c] for c in prefix] + [[121]] * n + [[122]], all_input=[0],
                      reporting=[k + n])


def report(state, at):
    return [(state << 32) | at]


def fastest(run, n=5):
    return min(run() for _ in range(n))


def test_plain_overflow_is_run_again_once(engine):
    # 16 waves' parts of a unit's worklist hold 16,384 items each, four waves' 65,536.
    # Run again on each call, the call took 1.47 times as long.
    n = 30000
    data = b"x" * 500 + b"ayz" + b"x" * 1000
    engine.load_groups([fan(n, b"a")], 1)
    engine.set_input(data, len(data))
    kw = dict(algorithm="nonblockinggroups", schedule="plain")
    print("[case] plain overflow", flush=True)
    engine.run(**kw)
    assert engine.reports().tolist() == report(n + 1, 502)
    again = fastest(lambda: engine.run(**kw)["kernel_ms"])
    four = fastest(lambda: engine.run(spill_capacity=65536, **kw)["kernel_ms"])
    assert engine.reports().tolist() == report(n + 1, 502)
    assert again < 1.2 * four, (again, four)


def test_noalloc_overflow_is_run_again_once(engine):
    # 390 workgroups have 3,697 items a wave in the scratch array, 78 have 18,480
    n = 10000
    data = np.full(200000, ord("x"), np.uint8)
    data[150000:150005] = np.frombuffer(b"abcyz", np.uint8)
    engine.load_groups([fan(n)], 3)
    opts = engine.options(schedule="batched", precompute_depth=3)
    small = engine.options(schedule="batched", precompute_depth=3, persistent_blocks=78)

    def run(o):
        got, st = run_noalloc(engine, o, data, data.size)
        assert got.tolist() == report(n + 3, 150004) and st.reports_raw == n
        return st.kernel_ms

    print("[case] noalloc overflow", flush=True)
    run(opts)
    again, few = fastest(lambda: run(opts)), fastest(lambda: run(small))
    assert again < 1.4 * few, (again, few)


# The all-group kernels: k_scan at depth 3, the general one at depth 2 and where the
# image has short reports.
KERNELS = [(3, False), (3, True), (2, False)]


def rule_set(n, short):
    # two automata that fan out, one that does not, and perhaps a two-byte report
    gs = [fan(n), fan(60, b"abq"), make_group(4, [(0, 1), (1, 2), (2, 3)], [[120]] * 4,
                                              all_input=[0], reporting=[3])]
    if short:
        gs.append(make_group(2, [(0, 1)], [[97], [98]], all_input=[0], reporting=[1]))
    return gs


def text(places, size=200000):
    data = np.full(size, ord("x"), np.uint8)
    for at in places:
        data[at:at + 5] = np.frombuffer(b"abcyz", np.uint8)
    data[77:82] = np.frombuffer(b"abqyz", np.uint8)
    return data


def expected(groups, data, chunk):
    return oracle.run(groups, data, chunk)[0]


@pytest.mark.parametrize("depth,short", KERNELS)
def test_overflow_marks_and_fallback(engine, depth, short):
    groups = rule_set(5000, short)
    chunk = 50000
    data = text([20, 25000, 99000, 149990, 160000])
    want = expected(groups, data, chunk)
    assert (want == report(5003, 24)[0]).sum() == 1
    engine.load_groups(groups, depth)
    engine.set_input(data, chunk)
    for unique in (False, True):
        kw = dict(schedule="batched", precompute_depth=depth, spill_capacity=64,
                  ring_capacity=64, window=512, unique=unique)
        print("[case] overflow", depth, short, unique, flush=True)
        with pytest.raises(NgapError) as e:
            engine.run(**kw)
        assert e.value.code == 4 and e.value.stats["overflow_units"] >= 4
        # 64 items x 16 x 16 hold them: two rounds of re-runs
        st = engine.run(fallback=True, **kw)
        assert st["fallback_tasks"] >= 2 * 4 and st["overflow_units"] >= 4
        assert np.array_equal(engine.reports(), want)
        # the caller's own work items
        tasks = [(-1, c, a, min(a + 700, chunk)) for c in range(4) for a in range(0, chunk, 700)]
        st = engine.run(fallback=True, tasks=tasks, **dict(kw, window=0))
        assert st["fallback_tasks"] > 0
        assert np.array_equal(engine.reports(), want)
        st = engine.run(schedule="batched", precompute_depth=depth, unique=unique)
        assert st["overflow_units"] == 0 and np.array_equal(engine.reports(), want)


@pytest.mark.parametrize("depth,short", KERNELS)
@pytest.mark.parametrize("n", [40000, 70000])
def test_small_jobs_retry_with_the_largest_worklists(engine, depth, short, n):
    # 200,000 positions: a wave's first worklist has 13,107 items, then 65,536
    groups, data = rule_set(n, short), text([150000])
    want = expected(groups, data, data.size)
    engine.load_groups(groups, depth)
    engine.set_input(data, data.size)
    kw = dict(schedule="batched", precompute_depth=depth)
    for turn in range(2):
        print("[case] retry", depth, short, n, turn, flush=True)
        if n < 65536:
            st = engine.run(**kw)
            assert st["overflow_units"] == 0 and st["fallback_tasks"] == 0
        else:
            with pytest.raises(NgapError) as e:
                engine.run(**kw)
            assert e.value.code == 4
            st = engine.run(fallback=True, **kw)
            assert st["fallback_tasks"] > 0
        assert st["reports_raw"] >= n
        assert np.array_equal(engine.reports(), want)


@pytest.mark.parametrize("depth,short", KERNELS)
def test_noalloc_on_the_smaller_grid(engine, depth, short):
    groups, data = rule_set(10000, short), text([150000])
    want = expected(groups, data, data.size)
    engine.load_groups(groups, depth)
    opts = engine.options(schedule="batched", precompute_depth=depth)
    for turn in range(2):
        print("[case] noalloc", depth, short, turn, flush=True)
        got, st = run_noalloc(engine, opts, data, data.size)
        assert np.array_equal(got, want) and st.overflow_units == 0


@pytest.mark.parametrize("depth", [1, 2, 3])
def test_plain_units_by_depth(engine, depth):
    # at depth 2 and 3 too: fewer waves after an overflow, then an error
    groups, data = rule_set(30000, True), text([500], 3000)
    want = expected(groups, data, data.size)
    engine.load_groups(groups, depth)
    engine.set_input(data, data.size)
    kw = dict(schedule="plain", precompute_depth=depth)
    print("[case] plain", depth, flush=True)
    for _ in range(2):
        st = engine.run(**kw)
        assert st["overflow_units"] == 0 and np.array_equal(engine.reports(), want)
    with pytest.raises(NgapError) as e:
        engine.run(spill_capacity=64, **kw)
    assert e.value.code == 4
    engine.run(**kw)
    assert np.array_equal(engine.reports(), want)


@pytest.mark.parametrize("schedule", ["plain", "batched"])
def test_counters_between_runs_of_the_default_algorithm(engine, schedule):
    groups, chunk = rule_set(2000, False), 50000
    data = text([20, 25000, 99000, 149990, 160000])
    want = expected(groups, data, chunk)
    engine.load_groups(groups, 3)
    engine.set_input(data, chunk)
    small = dict(spill_capacity=64, ring_capacity=64)
    first = {}
    steps = [dict(), dict(window=100), dict(), dict(over=True, **small), dict(),
             dict(fallback=True, **small), dict(window=100), dict(root_pass=True), dict(),
             dict(precompute_depth=2), dict(use_graph=True), dict(), dict(use_graph=True)]
    for k, kw in enumerate(steps):
        kw = dict(dict(precompute_depth=3), **kw)
        over = kw.pop("over", False)
        print("[case] counters", schedule, k, kw, flush=True)
        try:
            st = engine.run(schedule=schedule, **kw)
        except NgapError as e:
            assert (over or (schedule == "plain" and "spill_capacity" in kw)) and e.code == 4
            continue
        assert not over
        assert np.array_equal(engine.reports(), want)
        if "spill_capacity" in kw:
            continue  # (what is counted twice depends on which re-runs there were)
        counts = first.setdefault(tuple(sorted(kw.items())), (st["reports_raw"], st["items"]))
        assert counts == (st["reports_raw"], st["items"])
