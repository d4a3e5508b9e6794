"""Which step an engine takes (Engine.step_info) under every rule that chooses
one, each checked bit for bit against the CPU oracle in the same run: direct
propagation for all instances or none, its rounds of listed rows, the queue
tiles and the sharing of tiles from which rows are binned in a launch of their
own, and the settings that take either off."""
import numpy as np
import pytest

from test_direct import LIMIT, reorder
from test_gpu_parity import DT, assert_state_equal, run_oracle

pytestmark = pytest.mark.gpu

QUEUES = ("tile_bin", "bin_launch")


def add(dtb, eng, net, seed, mu):
    b = dtb.Block(net, delta_t=DT, seed=seed, engine=eng)
    b.update_ou_background_stimuli(b.subblk_id, 4.0, mu, 0.1)
    eng.configure(b.inst, 1, True)
    return b


def assert_oracle(orc, net, blk, steps, seed, mu):
    ref, sim = run_oracle(orc, net, steps, seed, mu)
    events = int((ref["raster"].astype(np.int64) * np.diff(net.rowptr)[None, :]).sum())
    assert events > 0 and blk.counters() == (steps, events, int(ref["raster"].sum()))
    assert_state_equal(blk.state(), sim)


def reversed_rows(dtb, net):
    """Rows by descending target: direct propagation is not allowed."""
    return reorder(dtb, net, -net.col.astype(np.int64))


@pytest.mark.parametrize("settings,mode", [
    ({}, "direct"),
    (dict(schedule=dict(layout="dense")), "tile_bin"),
    (dict(schedule=dict(layout="spread")), "tile_bin"),
    (dict(schedule=dict(pass_k=1, layout="auto")), "direct"),
    (dict(schedule=dict(layout="gather")), "gather"),
    (dict(split=dict(on=True)), "bin_launch"),
    (dict(split=dict(on=True, capacity=3)), "bin_launch"),
    (dict(pull=dict(on=False)), "tile_bin"),
    (dict(pull=dict(defer_min=1)), "tile_bin"),
    (dict(queue_capacity=dict(floor=64, shift=4)), "tile_bin"),
])
def test_mode_by_settings(dtb, orc, gpu, settings, mode):
    net, steps = dtb.gen_uniform(5000, 60, seed=4), 150
    eng = dtb.Engine(0)
    try:
        for name, kw in settings.items():
            getattr(eng, name)(**kw)
        b = add(dtb, eng, net, 3, 2.0)
        eng.run(steps, graph_chunk=50)
        assert eng.step_info()["mode"] == mode
        assert_oracle(orc, net, b, steps, 3, 2.0)
    finally:
        eng.close()


@pytest.mark.parametrize("n,mode", [(2, "direct"), (255, "direct"), (257, "direct"), (LIMIT, "direct"),
                                    (LIMIT + 1, "tile_bin")])
def test_direct_by_size(dtb, orc, gpu, n, mode):
    net, steps = dtb.gen_uniform(n, min(180, n - 1), seed=2), 40
    eng = dtb.Engine(0)
    try:
        b = add(dtb, eng, net, 13, 5.0)
        eng.run(steps)
        assert eng.step_info()["mode"] == mode
        assert_oracle(orc, net, b, steps, 13, 5.0)
    finally:
        eng.close()


def test_direct_for_all_instances_or_none(dtb, orc, gpu):
    """Unequal instances step directly; one that does not allow it takes all
    of them to queues, and back when it leaves, with spikes pending."""
    nets = [dtb.gen_uniform(3000, 60, seed=4), dtb.gen_voxel(30000, 12, 150, seed=3), dtb.gen_uniform(257, 20, seed=9)]
    other = reversed_rows(dtb, dtb.gen_uniform(9000, 120, seed=2))
    eng = dtb.Engine(0)
    try:
        blks = [add(dtb, eng, net, 70 + i, 2.0) for i, net in enumerate(nets)]
        eng.run(120, graph_chunk=50)
        assert eng.step_info()["mode"] == "direct"
        guest = add(dtb, eng, other, 90, 2.0)
        eng.run(101, graph_chunk=50)
        assert eng.step_info()["mode"] == "tile_bin"
        assert_oracle(orc, other, guest, 101, 90, 2.0)
        eng.remove(guest.inst)
        eng.run(60, graph_chunk=50)
        assert eng.step_info()["mode"] == "direct"
        for i, net in enumerate(nets):
            assert_oracle(orc, net, blks[i], 281, 70 + i, 2.0)
    finally:
        eng.close()


@pytest.mark.parametrize("rate", [0.04, 0.085])
def test_direct_rows_in_rounds(dtb, orc, gpu, rate):
    """More rows than a tile lists at a time (2048), and fewer than from which
    reading the in-edges is cheaper: two and three rounds in every step."""
    g = tuple(np.asarray(dtb.DEFAULT_G_UI) * 0.002)
    net, steps = dtb.gen_uniform(70_001, 400, seed=6, g_ui=g), 24
    net.props[:, 0] = rate   # noise spikes per step
    ref, sim = run_oracle(orc, net, steps, 19, 0.0, use_ou=False)
    rows = ref["raster"].sum(axis=1)
    edges = np.bincount(net.col >> 8, minlength=(net.n + 255) // 256).astype(np.float64)
    pulls_from = 12 * edges * net.n / (64.0 * net.n + 24 * edges)
    assert rows.min() > 2048 and rows.max() <= pulls_from.min()
    eng = dtb.Engine(0)
    try:
        b = dtb.Block(net, delta_t=DT, seed=19, engine=eng)
        out = b.run(steps, freqs=True, iou=False)
        assert eng.step_info()["mode"] == "direct" and eng.propagation_stats()["pulled"] == 0
        assert np.array_equal(out["freq"].sum(axis=1), rows)
        assert_state_equal(b.state(), sim)
    finally:
        eng.close()


@pytest.mark.parametrize("kind,n,mode", [("voxel", 3071 * 256, "tile_bin"), ("voxel", 3071 * 256 + 1, "bin_launch"),
                                         ("uniform", 3071 * 256 + 1, "tile_bin"),
                                         ("small voxels", 3072 * 256, "tile_bin")])
def test_binning_launch_by_tiles_and_sharing(dtb, orc, gpu, kind, n, mode):
    """From 3072 tiles, and only where rows have two synapses per tile they
    reach (uniform ones have one) and share these with the rows that fire
    beside them (voxels of 196 neurons share none)."""
    net = dtb.gen_uniform(n, 12, seed=5) if kind == "uniform" else \
        dtb.gen_voxel(n, 78 if kind == "voxel" else 4000, 220 if kind == "voxel" else 100, seed=6)
    rows = np.random.default_rng(1).integers(0, n, 300)
    seg = np.mean([len(np.unique(net.col[net.rowptr[r]:net.rowptr[r + 1]] >> 8)) for r in rows])
    assert (2.0 * seg <= net.nsyn / n) == (kind != "uniform")
    steps, mu = (40, 6.0) if kind == "uniform" else (24, 9.0)
    eng = dtb.Engine(0)
    try:
        b = add(dtb, eng, net, 40, mu)
        eng.run(steps)
        assert eng.step_info()["mode"] == mode
        assert_oracle(orc, net, b, steps, 40, mu)
    finally:
        eng.close()


def test_pass_lists_returned_in_direct_propagation(dtb, gpu):
    """The lists of the binning launch (131 kB here) go back when the engine
    turns to direct propagation."""
    eng = dtb.Engine(0)
    try:
        add(dtb, eng, dtb.gen_uniform(257, 20, seed=9), 3, 2.0)
        eng.split(True)
        eng.run(5)
        assert eng.step_info()["mode"] == "bin_launch"
        before = dtb.device_memory_cached(0)
        eng.split(False)
        eng.run(5)
        assert eng.step_info()["mode"] == "direct"
        assert dtb.device_memory_cached(0) - before > 64 * 1024
    finally:
        eng.close()


def test_offsets_that_do_not_fit_are_tried_once(dtb, gpu):
    """Where the offsets of one instance do not fit (313 MB, from a
    reservation with 64 MB left), the engine keeps queues and does not build
    and return those of the others at every run; it tries again when the
    instances change."""
    def fill(eng):
        small = dtb.Block(dtb.gen_uniform(3000, 60, seed=4), delta_t=DT, seed=3, engine=eng)
        return small, eng.add_fanout(200_000, 150, 5)

    dtb.device_memory_trim()
    dtb.device_memory_reserve(4 << 30)
    eng = dtb.Engine(0)
    try:
        eng.schedule(layout="dense")
        free = dtb.device_memory_cached(0)
        fill(eng)
        eng.run(2)
        used = free - dtb.device_memory_cached(0)
    finally:
        eng.close()
    dtb.device_memory_trim()
    dtb.device_memory_reserve(used + (64 << 20))
    eng = dtb.Engine(0)
    try:
        small, big = fill(eng)
        small.run(3, freqs=True)
        assert eng.step_info()["mode"] == "tile_bin"
        built = eng.step_info()["tables_built"]
        for _ in range(4):
            small.run(3, freqs=True)
        assert eng.step_info() == {"mode": "tile_bin", "tables_built": built}
        eng.remove(big)
        small.run(3, freqs=True)
        assert eng.step_info() == {"mode": "direct", "tables_built": built + 1}
    finally:
        eng.close()
        dtb.device_memory_trim()


def test_direct_stays_past_the_tiles_it_starts_from(dtb, gpu):
    """8192 tiles to start, 10240 to leave: an instance that comes and goes at
    8,200 tiles does not make the others' offsets go and come back."""
    n, k = 25_600, 30   # 100 tiles each
    eng = dtb.Engine(0)
    try:
        ids = [eng.add_fanout(n, k, 7 + i) for i in range(81)]
        eng.run(2)
        assert eng.step_info() == {"mode": "direct", "tables_built": 81}
        for turn in range(3):
            extra = eng.add_fanout(n, k, 500 + turn)
            eng.run(2)
            assert eng.step_info() == {"mode": "direct", "tables_built": 82 + turn}
            eng.remove(extra)
            eng.run(2)
            assert eng.step_info() == {"mode": "direct", "tables_built": 82 + turn}
        ids += [eng.add_fanout(n, k, 600 + i) for i in range(22)]
        eng.run(2)
        assert eng.step_info()["mode"] == "tile_bin"   # 10300 tiles
        for i in ids[90:]:
            eng.remove(i)
        eng.run(2)
        assert eng.step_info()["mode"] == "tile_bin"   # 9000: not from here
        for i in ids[81:90]:
            eng.remove(i)
        eng.run(2)
        assert eng.step_info()["mode"] == "direct"
    finally:
        eng.close()


@pytest.mark.parametrize("n,k", [(257, 20), (20_000, 100)])
def test_offsets_built_when_an_instance_is_added(dtb, orc, gpu, n, k):
    """Before its first step, beside the steps of the others; in memory that
    other data filled before (rows of no synapses among them)."""
    old = dtb.Engine(0)
    add(dtb, old, dtb.gen_uniform(n, 2 * k, seed=8), 5, 9.0)
    old.run(60)
    old.close()
    net = dtb.gen_uniform(n, k, seed=4)
    keep = np.repeat(np.arange(n), np.diff(net.rowptr)) % 5 != 0
    pre = np.repeat(np.arange(n), np.diff(net.rowptr))[keep]
    net = dtb.NetworkArrays.from_edges(net.props, pre, net.col[keep], net.w[keep], net.kind_per_synapse()[keep])
    eng = dtb.Engine(0)
    try:
        b = add(dtb, eng, net, 3, 3.0)
        assert eng.step_info()["tables_built"] == 1
        eng.run(100, graph_chunk=20)
        assert eng.step_info() == {"mode": "direct", "tables_built": 1}
        assert_oracle(orc, net, b, 100, 3, 3.0)
    finally:
        eng.close()


def test_autotuner_compares_the_binning_launch_with_binning_in_tiles(dtb, orc, gpu):
    """3072 tiles of a voxel network, nearly silent: ("dense", 2) is the
    binning launch, every other queue schedule bins in the tiles, and what is
    kept is what was timed."""
    net = dtb.gen_voxel(3072 * 256, 78, 220, seed=6)
    steps = 30
    eng = dtb.Engine(0)
    try:
        b = add(dtb, eng, net, 40, 9.0)
        eng.run(steps)
        assert eng.step_info()["mode"] == "bin_launch"
        for _ in range(4):
            k, layout, us = eng.autotune(16)
            print(k, layout, us, flush=True)
            eng.run(2)
            steps += eng.autotune_steps(16) + 2
            assert eng.step_info()["mode"] == ("gather" if layout == "gather" else
                                               "bin_launch" if (layout, k) == ("dense", 2) else "tile_bin")
        eng.schedule(layout="auto")
        eng.run(2)
        assert eng.step_info()["mode"] == "bin_launch"
        assert b.counters()[0] == steps + 2
    finally:
        eng.close()


def test_offsets_are_tried_again_when_memory_is_free(dtb, gpu):
    """The offsets of 313 MB do not fit beside another engine's instance; once
    that is gone, the next run steps directly."""
    def big(eng):
        b = dtb.Block(None, delta_t=DT, engine=eng, inst=eng.add_fanout(200_000, 150, 5))
        b.run(3, freqs=True)
        return b

    def guest(eng):
        eng.schedule(layout="dense")
        eng.add_fanout(100_000, 150, 6)
        eng.run(1)

    used = []
    for what in (guest, lambda e: (e.schedule(layout="dense"), big(e))):
        dtb.device_memory_trim()
        dtb.device_memory_reserve(4 << 30)
        eng = dtb.Engine(0)
        try:
            free = dtb.device_memory_cached(0)
            what(eng)
            used.append(free - dtb.device_memory_cached(0))
        finally:
            eng.close()
    dtb.device_memory_trim()
    dtb.device_memory_reserve(sum(used) + (64 << 20))
    other, eng = dtb.Engine(0), dtb.Engine(0)
    try:
        # the guest last, so that its range and the free one beside it are one
        eng.schedule(layout="dense")
        b = big(eng)
        guest(other)
        eng.schedule(layout="auto")
        for _ in range(3):
            b.run(3, freqs=True)
            assert eng.step_info()["mode"] == "tile_bin"
        other.close()
        other = None
        b.run(3, freqs=True)
        assert eng.step_info()["mode"] == "direct"
    finally:
        if other:
            other.close()
        eng.close()
        dtb.device_memory_trim()
