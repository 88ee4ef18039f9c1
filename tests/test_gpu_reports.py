"""Reports sorted on the device: sizes around the rank sort's wave, tile and
limit and the radix sort above it, with and without repeats, against the
reports the automaton gives by construction."""
import numpy as np
import pytest

from ngap_amd.groups import make_group

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1024, 1025, 8191, 16383, 16384, 16385, 40000])
@pytest.mark.parametrize("repeats", [False, True])
def test_sorted_unique_reports(engine, n, repeats):
    # every 'b' after an 'a' is reported: once, or once per all-input state
    starts = 2 if repeats else 1
    g = make_group(starts + 1, [(v, starts) for v in range(starts)],
                   [[ord("a")]] * starts + [[ord("b")]], all_input=range(starts),
                   reporting=[starts])
    print("[case] reports", n, repeats, flush=True)
    engine.load_groups([g], 1)
    engine.set_input(b"ab" * n, 2 * n)
    st = engine.run(schedule="batched", unique=False)
    want = (np.uint64(starts) << np.uint64(32)) | (2 * np.arange(n, dtype=np.uint64) + np.uint64(1))
    assert st["reports_raw"] == n * starts
    for _ in range(2):  # the second call copies what the first one sorted
        assert np.array_equal(engine.reports(), want)
