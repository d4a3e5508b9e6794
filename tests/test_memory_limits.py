"""What needs device memory only to be faster gives way where memory is short:
the same calls work as without it, with the same results.  The limits are
reservations of an exact size (blocks over 64 MB come from them or not at
all)."""
import numpy as np
import pytest

from test_gpu_parity import bits

pytestmark = pytest.mark.gpu


@pytest.fixture
def limit(dtb):
    """limit(fill, extra): reserves what fill(engine) takes, and `extra`
    bytes more."""
    def reserve(fill, extra):
        dtb.device_memory_trim()
        dtb.device_memory_reserve(8 << 30)
        eng = dtb.Engine(0)
        try:
            free = dtb.device_memory_cached(0)
            fill(eng)
            used = free - dtb.device_memory_cached(0)
        finally:
            eng.close()
        dtb.device_memory_trim()
        dtb.device_memory_reserve(used + extra)
    yield reserve
    dtb.device_memory_trim()


def test_gather_takes_larger_groups(dtb, gpu, limit):
    """250,000 neurons: offsets of 123 MB by groups of 1024 and 62 MB by
    groups of 2048; the records (600 MB) fit only beside the latter."""
    n, k, steps = 250_000, 200, 60

    def fill(eng, layout="dense"):
        eng.schedule(layout=layout)
        eng.pull(False)
        b = dtb.Block(None, delta_t=0.1, engine=eng, inst=eng.add_fanout(n, k, 5, seed=3))
        b.update_ou_background_stimuli(b.subblk_id, 4.0, 5.0, 0.1)
        eng.configure(b.inst, 1, True)
        eng.run(steps)
        return b

    limit(fill, 12 * n * k + (100 << 20))
    got = []
    for layout in ("gather", "dense"):
        eng = dtb.Engine(0)
        try:
            b = fill(eng, layout)
            assert eng.propagation(b.inst)["in_use"] == (layout == "gather")
            got.append((b.counters(), b.state()))
        finally:
            eng.close()
    assert got[0][0] == got[1][0] and got[0][0][2] > 1000
    for key in ("V", "J", "i_ou"):
        assert np.array_equal(bits(got[0][1][key]), bits(got[1][1][key])), key
