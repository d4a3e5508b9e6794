"""What a call does around its steps: parameters derived by several threads,
graphs kept from one call to the next while the tables they read change, and
records fetched in pieces.  Bit-exact against the CPU oracle, or against the
same steps in calls small enough to take one piece."""
import numpy as np
import pytest

from test_gpu_parity import DT, assert_state_equal, bits, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,values", [(40_001, 3), (40_001, 40_001), (70_000, 70_000)])
def test_parameters_of_ranges_of_neurons(dtb, orc, gpu, n, values):
    """Few classes that every thread's range meets in another order, one class
    per neuron, and more classes than the shared table takes."""
    net = dtb.gen_uniform(n, 40, seed=8)
    rng = np.random.default_rng(n)
    net.props[:, 18] *= (1.0 + rng.integers(0, values, n) / (4.0 * values)).astype(np.float32)
    net.props[rng.integers(0, n, 50), 1] = 1.0   # blocked
    out, st, cnt = run_gpu(dtb, net, 60, 23, 3.0, sample=np.array([0, n - 1], np.uint32))
    ref, sim = run_oracle(orc, net, 60, 23, 3.0)
    assert ref["raster"].sum() > 1000
    assert np.array_equal(out["freq"], ref["freq"])
    assert_state_equal(st, sim)


@pytest.mark.parametrize("layout", ["auto", "dense"])
def test_graphs_kept_while_tables_change(dtb, orc, gpu, layout):
    """Chunks of 64 graph steps over calls that change parameters, samples,
    statistics, the propagation settings and the set of instances."""
    net, other = dtb.gen_uniform(5000, 60, seed=4), dtb.gen_uniform(5000, 60, seed=5)
    ids = np.arange(0, 5000, 9, dtype=np.uint32)
    eng = dtb.Engine(0)
    freq, spikes = [], None
    try:
        eng.schedule(layout=layout)
        blk = dtb.Block(net, delta_t=DT, seed=3, engine=eng)
        blk.update_ou_background_stimuli(blk.subblk_id, 4.0, 2.0, 0.1)
        for turn in range(8):
            if turn == 2:
                blk.assign_property_by_subblk([1], [5], [-51.0])
            if turn == 3:
                blk.set_samples(ids)
            if turn == 5:
                eng.pull(True, 1)
            if turn == 6:
                b2 = dtb.Block(other, delta_t=DT, seed=9, engine=eng)
            if turn == 7:
                eng.remove(b2.inst)
            out = blk.run(130, graph=True, vmean=turn in (1, 4), output_sample_spike=turn >= 3)
            freq.append(out["freq"])
            spikes = out["spike"] if turn >= 3 else spikes
        st = blk.state()
        eng.check()
    finally:
        eng.close()
    on = orc.OracleNet.from_network(net, dt=DT, seed=3)
    on.set_ou(on.pop_ids, 2.0, 0.1, 4.0)
    sim = orc.Sim(on, 32)
    a = sim.run(260, raster=True, pop_counts=True)
    on.props[on.props[:, 3] == 1, 8] = -51.0
    b = sim.run(780, raster=True, pop_counts=True)
    assert a["raster"].sum() > 1000
    assert np.array_equal(np.concatenate(freq), np.concatenate([a["freq"], b["freq"]]))
    assert np.array_equal(spikes, b["raster"][-130:, ids])
    assert_state_equal(st, sim)


def test_record_fetched_in_pieces(dtb, gpu):
    """400 rows of 200 populations (4 MB) against the same steps in calls of
    40 rows, which fit one piece."""
    net = dtb.gen_voxel(20_000, 100, 60, seed=6)
    kw = dict(freqs=True, vmean=True, imean=True, receptor_imean=True)
    got = []
    for steps in (400, 40):
        blk = dtb.Block(net, delta_t=DT, seed=5)
        blk.update_ou_background_stimuli(blk.subblk_id, 4.0, 2.0, 0.1)
        outs = [blk.run(steps, **kw) for _ in range(400 // steps)]
        got.append({k: np.concatenate([np.asarray(o[k]) for o in outs], axis=1 if k == "receptor_imean" else 0)
                    for k in ("freq", "vmean", "imean", "receptor_imean")})
        blk.engine.close()
    assert got[0]["freq"].shape[1] == 200 and got[0]["freq"].sum() > 1000
    for k in got[0]:
        a, b = got[0][k], got[1][k]
        assert np.array_equal(a if k == "freq" else bits(a), b if k == "freq" else bits(b)), k
