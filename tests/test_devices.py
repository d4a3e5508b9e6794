"""An engine on one device, called by a thread that has another one current:
every call that allocates or launches makes its own device current first."""
import ctypes

import numpy as np
import pytest

from test_gpu_parity import DT, assert_state_equal, run_oracle

pytestmark = pytest.mark.gpu


def test_calls_with_another_device_current(dtb, orc, gpu):
    count = dtb.device_count()   # (with one device the calls are checked, and no switch)
    hip = ctypes.CDLL("libamdhip64.so")
    n, seed = 40_000, 7
    net = dtb.gen_uniform(n, 60, seed=4)
    eng = dtb.Engine(count - 1)
    try:
        b = dtb.Block(net, delta_t=DT, seed=seed, engine=eng)

        def other():
            assert hip.hipSetDevice(0) == 0

        other()
        b.update_ou_background_stimuli(b.subblk_id, 4.0, 3.0, 0.1)
        other()
        eng.configure(b.inst, 1, True)
        eng.run(60)
        other()
        b.assign_property_by_subblk([1], [5], [-51.0])   # THRESHOLD_V: new parameter records
        other()
        st = b.state()
        other()
        b.load_state(st)
        other()
        eng.run(60)
        other()
        st = b.state()
    finally:
        eng.close()
    on = orc.OracleNet.from_network(net, dt=DT, seed=seed)
    on.set_ou(on.pop_ids, 3.0, 0.1, 4.0)
    sim = orc.Sim(on, 32)
    a = sim.run(60, raster=True)
    on.props[on.props[:, 3] == 1, 8] = -51.0
    sim.run(60, raster=True)
    assert a["raster"].sum() > 1000
    assert_state_equal(st, sim)
    assert np.isfinite(st["V"]).all()
