"""The all-group scan kernel (memo depth 3, every report three symbols deep or
more): chunk lengths and windows around its 3-gram, its 128-position search
and its 8-byte loads, long lists of a slot, continuation records, start states,
repeats; against the oracle.  Shorter reports keep the general kernel."""
import random

import numpy as np
import pytest

import oracle
from ngap_amd.groups import make_group
from tests import nfa_helpers as H
from tests.test_zz_no_alloc import run_noalloc

pytestmark = pytest.mark.gpu

ALPHA = list(b"abc\xff")


def chain_rules(r, n, shortest):
    specs = [H.random_spec(r, r.randint(shortest, 6), ALPHA, p=(0.5, 0.4, 0.1), klo=2, khi=3)
             for _ in range(n)]
    return H.chains_group(specs)[0]


def fan_rules():
    # one 3-gram with 150 states behind it, each with nine successors (three
    # records), some of them shared; anchored states; a self-loop
    n = 3 + 150 + 9
    edges = [(0, 1), (1, 2)] + [(1, 3 + i) for i in range(150)]
    edges += [(3 + i, 153 + j) for i in range(0, 150, 7) for j in range(9)] + [(153, 153)]
    classes = [[97], [97, 98], [98]] + [[98, 99]] * 150 + [[97, 255]] * 5 + [range(256)] * 4
    return make_group(n, edges, classes, all_input=[0], start_of_data=[1],
                      reporting=list(range(150, n)))


@pytest.mark.parametrize("chunk", [1, 2, 3, 7, 8, 9, 63, 64, 65, 127, 128, 129, 130, 131, 1000])
@pytest.mark.parametrize("shortest", [2, 3])  # 2: reports at depth 2, the general kernel
def test_scan_edges(engine, chunk, shortest):
    r = random.Random(chunk)
    groups = [chain_rules(r, 6, shortest), fan_rules(), chain_rules(r, 2, 3)]
    for chunks in (1, 5):
        data = bytes(r.choice(ALPHA) for _ in range(chunk * chunks))
        engine.load_groups(groups, max_precompute_depth=3)
        engine.set_input(data, chunk, chunks)
        for dup in (False, True):
            want, _ = oracle.run(groups, data, chunk, chunks, is_dup=dup)
            for window in (0, 1, 64, 200):
                for unique in (False, True):
                    print("[case]", chunk, shortest, chunks, dup, window, unique, flush=True)
                    opts = engine.options(schedule="batched", precompute_depth=3, is_dup=dup,
                                          cross_groups=2, window=window, unique=unique)
                    engine.run(opts)
                    got = engine.reports()
                    assert np.array_equal(got, want), (got.size, want.size)
            got, _ = run_noalloc(engine, opts, np.frombuffer(data, np.uint8), chunk)
            assert np.array_equal(got, want), (got.size, want.size)


@pytest.mark.parametrize("blocks", [1, 3, 8, 9])  # below, at and above a queue an XCD
def test_work_item_claims(engine, blocks):
    # items a wave: below one, one, up to the last count that is all the
    # workgroups' own (six), just above it and far above
    r = random.Random(blocks)
    groups = [chain_rules(r, 4, 3), chain_rules(r, 2, 2), fan_rules()]
    chunk, chunks, waves = 997, 3, 4 * blocks
    data = bytes(r.choice(ALPHA) for _ in range(chunk * chunks))
    want, _ = oracle.run(groups, data, chunk, chunks)
    for depth in (2, 3):
        engine.load_groups(groups, max_precompute_depth=depth)
        engine.set_input(data, chunk, chunks)
        for items in (1, waves - 1, waves, waves + 1, 6 * waves - 1, 6 * waves, 6 * waves + 1,
                      40 * waves):
            window = max(1, -(-chunk // max(1, items // chunks)))
            for cross in (0, 2):
                print("[case] claims", blocks, depth, items, window, cross, flush=True)
                opts = engine.options(schedule="batched", precompute_depth=depth,
                                      cross_groups=cross, window=window,
                                      persistent_blocks=blocks)
                engine.run(opts)
                assert np.array_equal(engine.reports(), want)
                got, _ = run_noalloc(engine, opts, np.frombuffer(data, np.uint8), chunk)
                assert np.array_equal(got, want)
        # the program's own work items, of very different sizes
        cuts = [0] + sorted(r.sample(range(1, chunk), 5 * waves)) + [chunk]
        tasks = [(-1, c, a, b) for c in range(chunks) for a, b in zip(cuts, cuts[1:])]
        engine.run(schedule="batched", precompute_depth=depth, tasks=tasks,
                   persistent_blocks=blocks)
        assert np.array_equal(engine.reports(), want)
