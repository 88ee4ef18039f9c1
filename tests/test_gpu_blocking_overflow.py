"""blockinggroups' frontier at and just above its capacity: the states that do not
fit are in the last lanes of a wave, and the run must fail, not lose reports."""
import numpy as np
import pytest

from ngap_amd import NgapError
from ngap_amd.groups import make_group

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("states", [1, 63, 64, 65, 100, 255, 256, 257, 300])
@pytest.mark.parametrize("start", ["all-input", "start-of-data", "successors"])
def test_frontier_capacity(engine, states, start):
    # `states` states match at one position, and each one's successor reports at the next
    n = states
    edges, classes, first = [(i, n + i) for i in range(n)], [[97]] * n + [[98]] * n, range(n)
    data = b"xabx"
    if start == "successors":  # ... behind one state each
        edges += [(2 * n + i, i) for i in range(n)]
        classes += [[99]] * n
        first, data = range(2 * n, 3 * n), b"xcabx"
    starts = dict(all_input=first) if start != "start-of-data" else dict(start_of_data=first)
    if start == "start-of-data":
        data = data[1:]
    g = make_group(len(classes), edges, classes, reporting=range(n, 2 * n), **starts)
    at = data.index(b"b")
    want = (np.arange(n, 2 * n, dtype=np.uint64) << np.uint64(32)) | np.uint64(at)
    engine.load_groups([g], 1)
    engine.set_input(data, len(data))
    for cap in (n, n + 1, n - 1, max(0, n - 36)):
        if cap == 0:
            continue
        print("[case] blocking", states, start, cap, flush=True)
        if cap >= n:
            st = engine.run(algorithm="blockinggroups", spill_capacity=cap)
            assert st["overflow_units"] == 0
            assert np.array_equal(engine.reports(), want)
        else:
            with pytest.raises(NgapError) as e:
                engine.run(algorithm="blockinggroups", spill_capacity=cap)
            assert e.value.code == 4 and e.value.stats["overflow_units"] == 1
