"""Gather propagation at the sizes where its groups change (256 to 2048
neurons, at least 128 groups where the rows allow it) and with rows ordered
by groups of 2048 only: bit-exact against the CPU oracle."""
import numpy as np
import pytest

from test_gpu_parity import DT, assert_state_equal, bits, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,order", [(257, 30, "target"), (32_513, 40, "target"), (32_512, 40, "target"),
                                       (65_281, 40, "target"), (130_561, 40, "target"), (262_000, 40, "target"),
                                       (20_000, 7, "target"), (20_000, 40, "group")])
def test_gather_group_sizes(dtb, orc, gpu, n, k, order):
    net = dtb.gen_uniform(n, k, seed=n)
    if order == "group":
        pre = np.repeat(np.arange(n), np.diff(net.rowptr))
        o = np.lexsort((np.random.default_rng(2).random(net.nsyn), net.col >> 11, pre))
        net = dtb.NetworkArrays.from_edges(net.props, pre[o], net.col[o], net.w[o], net.kind_per_synapse()[o])
    ids = np.unique(np.r_[0, n - 1, np.arange(0, n, 101)]).astype(np.uint32)
    eng = dtb.Engine(0)
    try:
        eng.schedule(layout="gather")
        blk = dtb.Block(net, delta_t=DT, seed=7, engine=eng)
        assert eng.propagation(blk.inst)["in_use"]
        blk.update_ou_background_stimuli(blk.subblk_id, 4.0, 4.0, 0.1)
        blk.set_samples(ids)
        out = blk.run(70, graph=True, output_sample_spike=True, output_sample_isynaptic=True)
        st = blk.state()
        eng.check()
    finally:
        eng.close()
    ref, sim = run_oracle(orc, net, 70, 7, 4.0)
    assert ref["raster"].sum() > n // 4
    assert np.array_equal(out["freq"], ref["freq"])
    assert np.array_equal(out["spike"], ref["raster"][:, ids])
    assert_state_equal(st, sim)
    assert np.array_equal(bits(out["isynaptic"][-1]), bits(st["I_syn"][ids]))
