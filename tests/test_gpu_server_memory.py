"""A server's memory figures: what its launch buffers hold, to the byte, the list
of a launch's requests included, within a budget that leaves no room for more."""
import numpy as np
import pytest

from ngap_amd import synth
from ngap_amd.serve import FAILED, Server

pytestmark = pytest.mark.gpu

SPILL = 4 * 16384 * 8  # one workgroup's worklists


def window_of(total, waves=4):  # of the work items: a half of a wave's share
    w = 256
    while w < 4096 and 2 * w * waves < total:
        w *= 2
    return w


def launch_bytes(lens, window):
    total = sum(lens)
    items = sum(-(-n // window) for n in lens)
    return (total + 16 + (total // 32 + 2) * 4 + 32 * len(lens) +
            max(1 << 16, total // 2) * 8 + 24 * items + 4 * items + 4 + SPILL)


@pytest.mark.parametrize("lens", [[1], [1] * 3000, [300] * 700 + [5000]])
def test_held_bytes_cover_the_request_list(engine, lens):
    engine.load_groups([synth.regex_group(np.random.default_rng(1), 500)], 2)
    data = [np.full(n, 7, np.uint8) for n in lens]
    need = launch_bytes(lens, 256)  # admission counts the most work items there can be
    for budget in (need, need - 1):
        print("[case] server memory", len(lens), budget, flush=True)
        srv = Server(engine, budget_bytes=budget, max_inflight=1, precompute_depth=2,
                     algorithm="nonblockingallgroups", persistent_blocks=1)
        ids = [srv.submit(0, d) for d in data]
        while srv.pending() != (0, 0):
            srv.poll(block=True)
        st = srv.stats()
        assert st["peak_held_bytes"] <= budget
        if budget == need:
            assert st["launches"] == 1
            assert st["held_bytes"] == launch_bytes(lens, window_of(sum(lens)))
        elif len(lens) == 1:
            assert srv.take(ids[0])[0] == FAILED and st["rejected"] == 1
        else:
            assert st["rejected"] == 0 and st["launches"] > 1
        srv.close()
