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


@pytest.mark.parametrize("earlier", [False, True])
def test_samples_come_before_the_slots_of_the_sums(dtb, gpu, limit, earlier):
    """2000 rows of 10,000 samples (260 MB) fit with 16 MB to spare; the
    population sums' slots (33 MB), or those an earlier record left, must not
    take them first."""
    n, steps = 1 << 18, 2000
    ids = np.arange(0, n, 26, dtype=np.uint32)[:10_000]
    kw = dict(freqs=True, vmean=True, output_sample_spike=True, output_sample_vmemb=True, output_sample_isynaptic=True,
              output_sample_iou=True)

    def block(eng):
        b = dtb.Block(None, delta_t=0.1, engine=eng, inst=eng.add_fanout(n, 20, 5, seed=3))
        b.update_ou_background_stimuli(b.subblk_id, 4.0, 5.0, 0.1)
        b.set_samples(ids)
        b.run(1, freqs=True)
        return b

    limit(block, 13 * steps * ids.size + (16 << 20))
    eng = dtb.Engine(0)
    try:
        b = block(eng)
        if earlier:
            b.run(1000, freqs=True, vmean=True)
        got = b.run(steps, **kw)
    finally:
        eng.close()
    dtb.device_memory_trim()
    eng = dtb.Engine(0)
    try:
        b = block(eng)
        if earlier:
            b.run(1000, freqs=True, vmean=True)
        parts = [b.run(steps // 4, **kw) for _ in range(4)]
    finally:
        eng.close()
    assert got["freq"].sum() > 1000
    for key in ("freq", "vmean", "spike", "vmemb", "isynaptic", "iou"):
        want = np.concatenate([p[key] for p in parts])
        assert np.array_equal(bits(got[key]) if want.dtype == np.float32 else got[key],
                              bits(want) if want.dtype == np.float32 else want), key


def test_a_run_refused_for_its_record_leaves_none(dtb, gpu, limit):
    """A recorded run whose samples do not fit is refused; the steps after it
    record nothing, and a smaller record works."""
    n = 1 << 18
    ids = np.arange(0, n, 26, dtype=np.uint32)[:10_000]

    def block(eng):
        b = dtb.Block(None, delta_t=0.1, engine=eng, inst=eng.add_fanout(n, 20, 5, seed=3))
        b.update_ou_background_stimuli(b.subblk_id, 4.0, 5.0, 0.1)
        b.set_samples(ids)
        b.run(10, freqs=True)
        return b

    limit(block, 64 << 20)
    got = []
    for refused in (True, False):
        eng = dtb.Engine(0)
        try:
            b = block(eng)
            if refused:
                with pytest.raises(dtb.DtbError) as e:
                    b.run(4000, freqs=True, output_sample_vmemb=True)
                assert e.value.status == 101   # OUT_OF_MEMORY
            eng.run(100)
            got.append((b.run(60, freqs=True)["freq"], b.counters(), b.state()["V"]))
        finally:
            eng.close()
    assert got[0][0].sum() > 100 and np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]
    assert np.array_equal(bits(got[0][2]), bits(got[1][2]))
