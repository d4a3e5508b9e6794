"""Direct propagation (small instances with rows ordered by target: a tile
takes its input straight from the rows emitted in the step before) against
the CPU oracle, bit-exact, at the edges of its tiles, its row list, its
windows and its size limit; next to queue instances in one engine; and the
networks that do not allow it (rows not ordered by target, more neurons than
the limit), which keep the queues."""
import numpy as np
import pytest

from test_gpu_parity import DT, assert_state_equal, bits, run_oracle

pytestmark = pytest.mark.gpu

LIMIT = 1 << 18   # neurons up to which an instance propagates directly


def reorder(dtb, net, key):
    """net with each row's synapses in the order of key (per synapse)."""
    pre = np.repeat(np.arange(net.n), np.diff(net.rowptr))
    o = np.lexsort((key, pre))
    return dtb.NetworkArrays.from_edges(net.props, pre[o], net.col[o], net.w[o], net.kind_per_synapse()[o])


def ragged(dtb):
    """Rows of 0, of about 30 and of 60000 synapses on 20000 neurons."""
    n = 20000
    base = dtb.gen_uniform(n, 30, seed=3)
    rng = np.random.default_rng(5)
    pre = np.repeat(np.arange(n), np.diff(base.rowptr))
    keep = pre % 3 != 1
    hubs = np.array([0, 7, 255, 256, n - 1])
    hub_post = np.repeat(np.arange(n), 3)
    src = rng.integers(0, base.nsyn, len(hubs) * len(hub_post))
    pre2 = np.r_[pre[keep], np.repeat(hubs, len(hub_post))]
    post2 = np.r_[base.col[keep], np.tile(hub_post, len(hubs))]
    w2 = np.r_[base.w[keep], base.w[src] * np.float32(0.25)]
    k2 = np.r_[base.kind_per_synapse()[keep], base.kind_per_synapse()[src]]
    o = np.lexsort((post2, pre2))
    return dtb.NetworkArrays.from_edges(base.props, pre2[o], post2[o], w2[o], k2[o])


def check(dtb, orc, net, steps, seed, mu, layout="auto", pull=None, graph=False):
    ids = np.unique(np.r_[0, net.n - 1, np.arange(0, net.n, 97)]).astype(np.uint32)
    eng = dtb.Engine(0)
    try:
        eng.schedule(layout=layout)
        if pull is not None:
            eng.pull(pull)
        blk = dtb.Block(net, delta_t=DT, seed=seed, engine=eng)
        blk.update_ou_background_stimuli(blk.subblk_id, 4.0, mu, 0.1)
        blk.set_samples(ids)
        kw = dict(freqs=True, output_sample_spike=True, output_sample_vmemb=True, output_sample_isynaptic=True)
        a = blk.run(steps, **kw)
        eng.schedule(layout="dense" if layout == "auto" else "auto")   # the other path, with spikes pending
        b = blk.run(3, **kw)
        eng.schedule(layout=layout)
        c = blk.run(steps // 2, graph=graph, **kw)
        st, cnt, stats = blk.state(), blk.counters(), eng.propagation_stats()
        eng.check()
    finally:
        eng.close()
    total = steps + 3 + steps // 2
    ref, sim = run_oracle(orc, net, total, seed, mu, vtrace=True)
    for key, want in (("spike", ref["raster"][:, ids]), ("vmemb", ref["V"][:, ids]), ("freq", ref["freq"])):
        got = np.concatenate([a[key], b[key], c[key]])
        assert np.array_equal(bits(got) if key == "vmemb" else got, bits(want) if key == "vmemb" else want), key
    events = int((ref["raster"].astype(np.int64) * np.diff(net.rowptr)[None, :]).sum())
    assert cnt == (total, events, int(ref["raster"].sum()))
    assert_state_equal(st, sim)
    assert np.array_equal(bits(c["isynaptic"][-1]), bits(st["I_syn"][ids]))
    return ref["raster"].sum(axis=1), stats


@pytest.mark.parametrize("layout", ["auto", "dense"])
@pytest.mark.parametrize("n,k", [(2, 1), (255, 20), (256, 20), (257, 20), (5000, 40)])
def test_direct_tile_edges(dtb, orc, gpu, n, k, layout):
    rows, _ = check(dtb, orc, dtb.gen_uniform(n, k, seed=n), 300, 11, 1.5, layout, graph=True)
    assert rows.sum() > 0


@pytest.mark.parametrize("pull", [True, False])
@pytest.mark.parametrize("n,k,steps", [(66_049, 70, 120), (LIMIT, 180, 60), (LIMIT + 1, 180, 60)])
def test_direct_many_rows(dtb, orc, gpu, n, k, steps, pull):
    """From rest: the first volleys emit more rows than a tile lists at a
    time; with the in-edges it pulls, without it takes the rows in rounds."""
    rows, stats = check(dtb, orc, dtb.gen_uniform(n, k, seed=2), steps, 13, 5.0, pull=pull)
    assert rows.max() > 1024 and (rows > 0).sum() > 5
    assert (stats["pulled"] > 0) == pull or (pull and n > LIMIT)


@pytest.mark.parametrize("order", ["by target", "reversed"])
def test_direct_ragged_rows(dtb, orc, gpu, order):
    net = ragged(dtb)
    if order == "reversed":
        net = reorder(dtb, net, -net.col.astype(np.int64))   # does not allow direct propagation
    rows, _ = check(dtb, orc, net, 200, 17, 1.5)
    assert rows.sum() > 1000


def test_direct_and_queue_instances_in_one_engine(dtb, orc, gpu):
    a, c = dtb.gen_uniform(3000, 60, seed=4), dtb.gen_voxel(30000, 12, 150, seed=3)
    nets = [a, reorder(dtb, dtb.gen_uniform(9000, 120, seed=2), np.random.default_rng(1).random(9000 * 120)),
            c, reorder(dtb, c, -c.col.astype(np.int64)), dtb.gen_uniform(257, 20, seed=9)]
    steps, eng = 250, dtb.Engine(0)
    try:
        ids = []
        for i, net in enumerate(nets):
            b = dtb.Block(net, delta_t=DT, seed=70 + i, engine=eng)
            b.update_ou_background_stimuli(b.subblk_id, 4.0, 2.0, 0.1)
            eng.configure(b.inst, 1, True)
            ids.append(b)
        eng.run(steps, graph_chunk=50)
        got = [(b.state(), b.counters()) for b in ids]
        eng.check()
    finally:
        eng.close()
    for i, net in enumerate(nets):
        ref, sim = run_oracle(orc, net, steps, 70 + i, 2.0)
        events = int((ref["raster"].astype(np.int64) * np.diff(net.rowptr)[None, :]).sum())
        assert got[i][1] == (steps, events, int(ref["raster"].sum())), i
        assert_state_equal(got[i][0], sim)
