"""The bench line's measured traffic is only of the kernels that ran: a
profile of other kernels, or of other device code, gives none."""
import os

from test_bench_profiles import ROOT, WINDOW, load_bench


def test_traffic_only_for_the_profiled_kernels():
    bench = load_bench()
    for name in bench.PROFILES:
        lines = [x.strip() for x in open(os.path.join(ROOT, "profiles", name))]
        wl, n, layout, steps, warmup, tuned = next(m for m in map(WINDOW.match, lines) if m).groups()
        kernels = [x.split(": ", 1)[1] for x in lines if x.startswith("kernels: ")]
        source = [x.split(": ", 1)[1] for x in lines if x.startswith("device_source: ")]
        assert len(kernels) == 1 and kernels[0] in bench.STEP_KERNELS.values() and len(source) == 1, name
        window = (wl, int(n), layout, int(steps), int(warmup), tuned == "1")
        assert bench.profiled_traffic(*window, kernels[0], source[0])[1] == "profiles/" + name
        for other in bench.STEP_KERNELS.values():
            if other != kernels[0]:
                assert bench.profiled_traffic(*window, other, source[0]) == (None, None)
        assert bench.profiled_traffic(*window, kernels[0], "0" * 16) == (None, None)


def test_device_source_follows_the_code(tmp_path, monkeypatch):
    bench = load_bench()
    csrc = tmp_path / "digital_twin_brain-open_amd" / "csrc"
    csrc.mkdir(parents=True)
    for f in ("dtb_kernels.hip", "dtb_types.hpp", "dtb_rng.hpp"):
        (csrc / f).write_text(open(os.path.join(ROOT, "digital_twin_brain-open_amd", "csrc", f)).read())
    here = bench.device_source()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.device_source() == here
    text = (csrc / "dtb_rng.hpp").read_text()
    (csrc / "dtb_rng.hpp").write_text("// another comment\n" + text + "\n/* and\n one more */\n")
    assert bench.device_source() == here
    (csrc / "dtb_rng.hpp").write_text(text + "constexpr int more = 1;\n")
    assert bench.device_source() != here
