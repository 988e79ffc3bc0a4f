"""The plain PTT queue kernel at the sizes where its probe groups can go
wrong, bit-exact against the CPU oracle: probe counts around the groups of 8
whose taps are shared by the lanes, without corner blocks (every tap takes the
slow path), and a maximum length that ends passes on the last sub-step."""

import dataclasses

import pytest

from test_gpu_parity import _assert_same, _run_both

pytestmark = pytest.mark.gpu


def _check(w, n=10, seed=9, **kw):
    from gpustreamlines_amd import workloads as W

    seeds = W.seeds_for(w, n, placement="mixed", seed=seed)
    g, o = _run_both(w, seeds, **kw)
    assert len(o["sline_len"]) > 0
    _assert_same(g, o)


@pytest.mark.parametrize("blocks", [True, False])
@pytest.mark.parametrize("probes", [1, 2, 3, 7, 8, 9, 17])
def test_probe_counts(small_workloads, probes, blocks):
    w0 = small_workloads["ptt"]
    w = dataclasses.replace(w0, params=dict(w0.params, probe_quality=probes, max_sline_len=40))
    _check(w, blocks=blocks)


@pytest.mark.parametrize("frac,maxlen", [(1, 9), (3, 9), (10, 2)])
def test_last_sub_step(small_workloads, frac, maxlen):
    w0 = small_workloads["ptt"]
    w = dataclasses.replace(w0, params=dict(w0.params, step_frac=frac, max_sline_len=maxlen))
    _check(w, n=24)
