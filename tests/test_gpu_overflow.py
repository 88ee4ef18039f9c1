"""Worklists that overflow, on the kernels of the default algorithm: what a run's
smaller default worklists cannot hold is run again with larger ones, once and not
on every call; against reports known by construction."""
import numpy as np
import pytest

from ngap_amd import Engine
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
