"""The bootstrap kernels' variant follows the seeds in flight on the card, not
those of one launch: a pipeline's handles each hold a chunk, and the 2-waves
variant on all of them leaves half of the card's slots unused."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _limit(dt):
    """Most seeds that a launch on this handle gives the 2-waves variant."""
    lo, hi = 1, 1 << 24
    assert dt.boot_waves(lo) == 2 and dt.boot_waves(hi) == 4
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if dt.boot_waves(mid) == 2 else (lo, mid)
    return lo


@pytest.mark.parametrize("mode", [0, 1])
def test_variant_by_seeds_in_flight(small_workloads, mode):
    from gpustreamlines_amd._device import DeviceTracker

    dt = DeviceTracker(small_workloads["csa"].params, device=0)
    forks = []
    try:
        dt.set_boot_mode(mode)
        alone = _limit(dt)
        for k in range(2, 9):
            forks.append(dt.fork())
            assert _limit(dt) == alone // k and all(_limit(f) == alone // k for f in forks)
        forks.pop().close()
        assert _limit(dt) == alone // 7
        dt.set_boot_mode(mode, 4)
        assert dt.boot_waves(1) == 4
        dt.set_boot_mode(mode, 2)
        assert dt.boot_waves(1 << 24) == 2
    finally:
        for f in forks:
            f.close()
        dt.close()


@pytest.mark.parametrize("kind,mode", [("csa", 0), ("opdt", 0), ("csa", 1), ("opdt", 1)])
def test_both_variants_give_the_same_streamlines(small_workloads, kind, mode):
    from gpustreamlines_amd import workloads as W
    from test_gpu_boot_mfma import _track

    w = small_workloads[kind]
    seeds = W.seeds_for(w, 300, placement="mixed", seed=2)
    a, b = (_track(w, seeds, mode, occ=occ) for occ in (2, 4))
    assert len(a["sline_len"]) > 0
    for k in ("counts", "sline_seed", "sline_len", "points"):
        assert np.array_equal(a[k], b[k]), k
