"""A request launch set up on the device: request lengths around the gather's
16-byte units, its 4 KiB per wave and the work items' windows, many requests in
one launch, equal lengths, more reports than the pinned ones; against the
oracle, request by request."""
import random

import numpy as np
import pytest

import oracle
from ngap_amd.groups import make_group
from ngap_amd.serve import Server
from tests import nfa_helpers as H

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 4095, 4096,
           4097, 8193, 65535, 65536, 65537]


@pytest.mark.parametrize("case", ["mixed", "one", "many", "dense"])
def test_requests_of_all_lengths(engine, case):
    r = random.Random(len(case))
    alpha = list(b"abc\x00")
    specs = [H.random_spec(r, r.randint(2, 5), alpha) for _ in range(8)]
    groups = [H.chains_group(specs[:4])[0], H.chains_group(specs[4:], start="start-of-data")[0],
              make_group(1, [], [alpha], all_input=[0], reporting=[0])]
    lens = {"mixed": LENGTHS * 2, "one": [70001], "many": [r.choice(LENGTHS[:12]) for _ in range(700)],
            "dense": [20000, 17, 16384]}[case]
    r.shuffle(lens)
    which = [2 if case == "dense" else r.randrange(2) for _ in lens]
    data = [np.frombuffer(bytes(r.choice(alpha) for _ in range(n)), np.uint8) for n in lens]
    engine.load_groups(groups, max_precompute_depth=3)
    srv = Server(engine, max_inflight=3, algorithm="nonblockingallgroups", schedule="batched",
                 precompute_depth=3)
    for turn in range(2):  # the second on buffers that the first one used
        print("[case] requests", case, turn, len(lens), flush=True)
        ids = [srv.submit(g, d) for g, d in zip(which, data)]
        done = srv.drain(ids)
        for i, g, d in zip(ids, which, data):
            want, _ = oracle.run([groups[g]], d.tobytes(), len(d), 1)
            # a request's reports carry its group's number
            want = want | (np.uint64(g) << np.uint64(54))
            assert np.array_equal(done[i][0], want), (case, g, len(d))
    srv.close()
