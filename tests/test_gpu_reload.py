"""Other groups loaded while a server has launches in flight and requests queued:
what was launched ends on the groups it was started with (a re-run of overflowed
work items too), what is queued is scanned with the new ones, a request whose
group is gone fails, and nothing is launched while no groups are loaded."""
import numpy as np
import pytest

import oracle
from ngap_amd import NgapError, synth
from ngap_amd.groups import Group, make_group
from ngap_amd.serve import FAILED, INFLIGHT, QUEUED, Server

pytestmark = pytest.mark.gpu


def rule_set(seed, n=4):
    rng = np.random.default_rng(seed)
    return [synth.regex_group(rng, 4000, dotstar=(i == 1)) for i in range(n)]


def expected(groups, g, data):
    want, _ = oracle.run([groups[g]], data, len(data), 1)
    return want | (np.uint64(g) << np.uint64(54))


def fan(n):
    # one "abcd" queues n items in one wave: more than a launch's worklist holds
    return make_group(n + 4, [(0, 1), (1, 2)] + [(2, 3 + i) for i in range(n)] +
                      [(3 + i, n + 3) for i in range(n)],
                      [[97], [98], [99]] + [[100]] * n + [[101]], all_input=[0],
                      reporting=[n + 3])


@pytest.mark.parametrize("overflow", [False, True])
def test_load_while_launches_are_in_flight(engine, overflow):
    old, new = rule_set(1), rule_set(2)  # images of about the same size
    rng = np.random.default_rng(3)
    reqs = [(i % 4, synth.zipf_bytes(rng, 1 << 20, 0.9)) for i in range(8)]
    if overflow:
        old[0] = fan(40000)
        for i in (0, 4):
            reqs[i][1][1000:1005] = np.frombuffer(b"abcde", np.uint8)
    engine.load_groups(old, 3)
    srv = Server(engine, max_inflight=2, algorithm="nonblockingallgroups", precompute_depth=3)
    print("[case] reload", overflow, flush=True)
    first = [srv.submit(g, d) for g, d in reqs]
    srv.poll()
    assert all(srv.take(i)[0] == INFLIGHT for i in first)
    later = [srv.submit(g, d) for g, d in reqs]
    assert all(srv.take(i)[0] == QUEUED for i in later)
    engine.load_groups(new, 3)
    assert srv.pending() == (len(later), 0)
    assert srv.stats()["redone"] >= (1 if overflow else 0)
    done = srv.drain(first + later)
    for i, j, (g, d) in zip(first, later, reqs):
        assert np.array_equal(done[i][0], expected(old, g, d)), (g, "before the load")
        assert np.array_equal(done[j][0], expected(new, g, d)), (g, "after the load")
    srv.close()


def test_queued_requests_after_loads(engine):
    old, new = rule_set(4, 4), rule_set(5, 2)
    data = synth.zipf_bytes(np.random.default_rng(6), 5000, 0.9)
    engine.load_groups(old, 2)
    srv = Server(engine, max_inflight=2, algorithm="nonblockingallgroups", precompute_depth=2)
    ids = [srv.submit(g, data) for g in range(4)]
    broken = Group(new[0].row, new[0].col.copy(), new[0].sets, new[0].attrs, new[0].aas,
                   new[0].sod)
    broken.col[0] = 1 << 20  # out of range
    print("[case] reload: no groups", flush=True)
    with pytest.raises(NgapError):
        engine.load_groups([broken], 2)
    with pytest.raises(NgapError):
        srv.poll()
    assert srv.pending() == (4, 0)
    engine.load_groups(new, 1)  # not the depth that the server asks for
    with pytest.raises(NgapError):
        srv.poll()
    print("[case] reload: fewer groups", flush=True)
    engine.load_groups(new, 2)
    done = srv.drain(ids[:2])
    for g in range(2):
        assert np.array_equal(done[ids[g]][0], expected(new, g, data))
    assert [srv.take(i)[0] for i in ids[2:]] == [FAILED, FAILED]
    # a server that outlives its launches' groups, closed after another load
    srv.submit(0, data)
    srv.poll()
    engine.load_groups(old, 2)
    srv.close()
    engine.load_groups(new, 2)
