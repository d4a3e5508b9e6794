"""The footprint that admission counts covers what an instance takes on the
device, and what the engine takes only where memory allows does not refuse a
request that fits without it."""
import importlib

import pytest

from test_serving_host import requests, serving   # noqa: F401 (fixture with a stand-in engine)


def test_a_request_that_fits_without_the_optional_tables_is_served(serving):  # noqa: F811
    reqs = requests(serving, 4)
    least = max(r.device_bytes(pull=True, optional=False) for r in reqs)
    assert least < min(r.device_bytes(pull=True) for r in reqs[-1:])
    srv = serving.Server(hbm_budget=least, chunk=100, reserve=False)
    stats = srv.serve(reqs, realtime=False)
    assert stats["shed"] == 0 and all(r.events == 7 * r.steps for r in reqs)
    assert srv.engine.max_resident == 1
    with pytest.raises(ValueError):
        serving.Server(hbm_budget=least - 1, chunk=100, reserve=False).serve(requests(serving, 4), realtime=False)


def test_optional_tables_are_counted(serving):  # noqa: F811
    """Offsets of direct propagation by the engine's conditions; pass lists
    otherwise; gather's groups of 256 to 2048 neurons."""
    def extra(n, k, **kw):
        r = serving.Request(0, 0.0, n, k, 10, 1, 1, 3.0)
        return r.device_bytes(**kw) - r.device_bytes(optional=False, **kw)

    lists = lambda n, k: 8 * 64 * -(-(-(-n // 256)) // 64) * 256 * -(-k // 256) + 2 * 64 * 32 * 4  # noqa: E731
    assert extra(200_000, 400, pull=True) == 2 * 200_000 * 783
    assert extra(1 << 18, 400, pull=True) == 2 * (1 << 18) * 1025
    assert extra((1 << 18) + 1, 400, pull=True) == lists((1 << 18) + 1, 400)
    assert extra(200_000, 400, pull=False) == lists(200_000, 400)
    assert extra(200_000, 50, pull=True) == lists(200_000, 50)   # offsets larger than the synapses
    assert extra(200_000, 400, gather=True) == 2 * 200_000 * (196 - 98)
    assert extra(30_000, 400, gather=True) == 2 * 30_000 * (118 - 15)
    assert extra(300_000, 400, gather=True) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["auto", "gather"])
@pytest.mark.parametrize("n,k", [(9000, 120), (60_000, 200), (200_000, 150), (300_000, 100)])
def test_footprint_covers_what_an_instance_takes(dtb, gpu, layout, n, k):
    mod = importlib.import_module("digital_twin_brain-open_amd.serving")
    r = mod.Request(0, 0.0, n, k, 10, 1, 1, 3.0)
    counted = r.device_bytes(layout == "gather", pull=True)
    dtb.device_memory_trim()
    srv = mod.Server(hbm_budget=4 << 30, layout=layout)
    try:
        srv.engine.run(0)
        free = dtb.device_memory_cached(0)
        srv._admit(r)
        srv.engine.run(2)
        srv.engine.sync()
        used = free - dtb.device_memory_cached(0)
        assert srv.engine.step_info()["mode"] == ("gather" if layout == "gather" else
                                                  "direct" if n <= 1 << 18 else "tile_bin")
        print(layout, n, k, used, counted, flush=True)
        # the engine's own tables: 4 KB blocks and about a byte per neuron
        assert used <= counted + n + (1 << 19)
    finally:
        srv.close()
        dtb.device_memory_trim()
