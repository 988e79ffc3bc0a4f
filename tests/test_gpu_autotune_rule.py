"""Tuning on a sample leaves the bootstrap kernel's variant to each launch's
seeds, and times the variant that the runs will take."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("run_seeds", [0, 1_000_000])
def test_tune_on_a_sample(small_workloads, mode, run_seeds):
    from gpustreamlines_amd import autotune
    from gpustreamlines_amd import workloads as W
    from gpustreamlines_amd._device import DeviceTracker

    w = small_workloads["csa"]
    seeds = W.seeds_for(w, 200, placement="mixed")
    dt = DeviceTracker(w.params, device=0)
    try:
        dt.upload(w.dataf, w.stop_map, w.vertices, w.edges, boot=w.boot)
        dt.set_boot_mode(mode)
        ref = dt.track(seeds)
        best, times = autotune.tune(dt, seeds, run_seeds=run_seeds)
        print(best, times, flush=True)
        assert tuple(sorted(best.items())) in times
        assert tuple(sorted(autotune.default(1, mode).items())) in times
        assert dt.boot_mode == mode
        assert not (run_seeds and best.get("waves_per_simd"))
        if not best.get("waves_per_simd"):
            assert dt.boot_waves(1) == 2 and dt.boot_waves(1 << 24) == 4
        got = dt.track(seeds)
    finally:
        dt.close()
    assert np.array_equal(ref["points"], got["points"]) and np.array_equal(ref["sline_len"], got["sline_len"])
