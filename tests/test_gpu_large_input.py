"""Large inputs: the default schedule's list of work items, made for every new
input, stays short, and the reports are those of short windows."""
import numpy as np
import pytest

from ngap_amd import Engine, synth
from ngap_amd.groups import make_group
from tests.test_zz_no_alloc import run_noalloc

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("size,chunk", [(64 * MIB, 64 * MIB), (256 * MIB, MIB),
                                        (300 * MIB + 7, 300 * MIB + 7), (256 * MIB, 4096)])
def test_work_items_of_large_inputs(size, chunk):
    rng = np.random.default_rng(1)
    groups = [synth.regex_group(rng, 400, dotstar=(i == 0)) for i in range(3)]
    part = synth.zipf_bytes(rng, 16 * MIB, 0.9)
    groups.append(make_group(4, [(0, 1), (1, 2), (2, 3)], [[int(b)] for b in part[1000:1004]],
                             all_input=[0], reporting=[3]))
    data = np.tile(part, -(-size // part.size))[:size]
    with Engine(0) as e:
        e.load_groups(groups, 3)
        e.set_input(data, chunk)
        print("[case] large input", size, chunk, flush=True)
        kw = dict(schedule="batched", precompute_depth=3)
        st = e.run(**kw)
        got = e.reports()
        assert st["num_tasks"] <= 65536 + size // chunk
        e.run(window=1024, **kw)
        assert got.size > 0 and np.array_equal(got, e.reports())
        got2, st2 = run_noalloc(e, e.options(**kw), data, chunk, cap=1 << 22)
        assert np.array_equal(got2, got)
        assert st2.num_tasks <= 65536 + size // chunk
