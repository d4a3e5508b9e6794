"""Binning by a launch of its own (split binning, and engines of many queue
tiles) against the CPU oracle, bit-exact: rows of no, one and many passes,
more target tiles than one window of the LDS counts holds, the size from
which it is taken, and instances of unequal size on one launch."""
import numpy as np
import pytest

from test_direct import ragged
from test_gpu_parity import DT, assert_state_equal, run_oracle

pytestmark = pytest.mark.gpu


def check(dtb, orc, nets, steps, mu, split=None, pull=None, queue=None, layout="auto"):
    eng = dtb.Engine(0)
    try:
        eng.schedule(layout=layout)
        if split is not None:
            eng.split(split)
        if pull is not None:
            eng.pull(pull)
        if queue is not None:
            eng.queue_capacity(*queue)
        blks = []
        for i, net in enumerate(nets):
            b = dtb.Block(net, delta_t=DT, seed=40 + i, engine=eng)
            b.update_ou_background_stimuli(b.subblk_id, 4.0, mu, 0.1)
            eng.configure(b.inst, 1, True)
            blks.append(b)
        eng.run(steps // 2 + 1)
        eng.run(steps - steps // 2 - 1, graph_chunk=10)
        got = [(b.state(), b.counters()) for b in blks]
        stats = eng.propagation_stats()
        eng.check()
    finally:
        eng.close()
    for i, net in enumerate(nets):
        ref, sim = run_oracle(orc, net, steps, 40 + i, mu)
        events = int((ref["raster"].astype(np.int64) * np.diff(net.rowptr)[None, :]).sum())
        assert events > 0 and got[i][1] == (steps, events, int(ref["raster"].sum())), i
        assert_state_equal(got[i][0], sim)
    return stats


@pytest.mark.parametrize("queue", [None, (64, 4)])
@pytest.mark.parametrize("pull", [True, False])
def test_rows_of_many_passes(dtb, orc, gpu, pull, queue):
    stats = check(dtb, orc, [ragged(dtb), dtb.gen_uniform(257, 300, seed=3)], 160, 2.0, True, pull, queue)
    assert queue is None or (stats["pulled"] if pull else stats["spilled"]) > 0


def test_more_tiles_than_one_window(dtb, orc, gpu):
    check(dtb, orc, [dtb.gen_uniform(16384 * 256 + 5, 3, seed=4)], 24, 9.0, True, False)


@pytest.mark.parametrize("n", [3071 * 256, 3071 * 256 + 1])
def test_size_from_which_it_is_taken(dtb, orc, gpu, n):
    check(dtb, orc, [dtb.gen_uniform(n, 12, seed=5)], 40, 6.0)


def test_taken_where_rows_share_tiles(dtb, orc, gpu):
    """A voxel network of 3072 tiles whose rows have two synapses per tile
    they reach (the uniform ones above have one)."""
    net = dtb.gen_voxel(3072 * 256, 78, 220, seed=6)
    rows = np.random.default_rng(1).integers(0, net.n, 500)
    seg = [len(np.unique(net.col[net.rowptr[r]:net.rowptr[r + 1]] >> 8)) for r in rows]
    assert 2.0 * np.mean(seg) < 0.98 * 220
    check(dtb, orc, [net], 24, 9.0)
