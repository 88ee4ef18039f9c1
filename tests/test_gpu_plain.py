"""The plain schedule's units on 4, 8 and 16 waves: few and many units, chunks
shorter than the waves' shares, a backlog that only four waves' worklists hold."""
import random

import numpy as np
import pytest

import oracle
from ngap_amd.groups import make_group
from tests import nfa_helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk,chunks", [(1, 1), (63, 1), (4097, 1), (70, 100), (33, 255),
                                          (33, 257), (17, 513), (5, 1300)])
@pytest.mark.parametrize("depth", [0, 1, 3])
def test_plain_units(engine, chunk, chunks, depth):
    r = random.Random(chunk)
    alpha = list(b"abc")
    groups = [H.chains_group([H.random_spec(r, r.randint(1, 5), alpha) for _ in range(4)],
                             start=s)[0] for s in ("all-input", "start-of-data")]
    data = bytes(r.choice(alpha) for _ in range(chunk * chunks))
    for dup in (False, True):
        want, _ = oracle.run(groups, data, chunk, chunks, is_dup=dup)
        engine.load_groups(groups, max(depth, 1))
        engine.set_input(data, chunk, chunks)
        print("[case] plain", chunk, chunks, depth, dup, flush=True)
        engine.run(schedule="plain", precompute_depth=depth, is_dup=dup)
        assert np.array_equal(engine.reports(), want)


def test_plain_backlog_of_one_wave(engine):
    # one position queues 30,000 items: more than a sixteenth of a unit's
    # worklist, less than a quarter
    n = 30000
    g = make_group(n + 2, [(0, 1 + i) for i in range(n)] + [(1 + i, n + 1) for i in range(n)],
                   [[97]] + [[98]] * n + [[99]], all_input=[0], reporting=[n + 1])
    engine.load_groups([g], 1)
    engine.set_input(b"xxabcxxx", 8)
    print("[case] plain backlog", flush=True)
    st = engine.run(algorithm="nonblockinggroups", schedule="plain")
    assert st["reports_raw"] == n and st["overflow_units"] == 0
    assert [int(x) for x in engine.reports()] == [((n + 1) << 32) | 4]


def test_batched_backlog_of_one_wave(engine):
    # the same on the batched schedule, whose small jobs have smaller worklists
    n = 40000
    g = make_group(n + 2, [(0, 1 + i) for i in range(n)] + [(1 + i, n + 1) for i in range(n)],
                   [[97]] + [[98]] * n + [[99]], all_input=[0], reporting=[n + 1])
    data = b"x" * 150000 + b"abc" + b"x" * 50000
    for depth in (1, 2, 3):
        engine.load_groups([g], depth)
        engine.set_input(data, len(data))
        print("[case] batched backlog", depth, flush=True)
        for _ in range(2):
            st = engine.run(algorithm="nonblockinggroups", schedule="batched",
                            precompute_depth=depth)
            assert st["reports_raw"] == n and st["overflow_units"] == 0
            assert [int(x) for x in engine.reports()] == [((n + 1) << 32) | 150002]
