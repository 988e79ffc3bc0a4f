"""The register-resident probabilistic kernel at the sizes and values where it
can go wrong, bit-exact against the CPU oracle: spheres around the chunk
boundaries (256 channels; rows of more than 768 channels take the general
kernel), steps that stay in a cell, cross one face or several and jump over
cells, flat volumes, symmetric spheres, and pmf values that leave the fast
path (NaN, infinities, negative and huge values)."""

import functools

import numpy as np
import pytest

from test_gpu_parity import _assert_same, _run_both

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=None)
def _sphere(n):
    from gpustreamlines_amd.sphere import symmetric_sphere

    return symmetric_sphere(n)


def _workload(nverts, shape=(13, 11, 12), step=0.3, symm=0, spoil=None, seed=5):
    from gpustreamlines_amd import workloads as W

    rng = np.random.default_rng(seed)
    verts, edges = _sphere(nverts)
    ax = np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1) / 6.0
    d = np.stack([np.cos(ax @ rng.normal(size=3) + k) for k in range(3)], -1)
    d /= np.linalg.norm(d, axis=-1, keepdims=True)
    odf = np.exp(6.0 * ((d @ verts.T.astype(np.float64)) ** 2 - 1.0)) + 0.02 * rng.random(shape + (nverts,))
    odf = np.ascontiguousarray(odf, dtype=np.float32)
    stop = np.ones(shape, np.float32)
    stop[rng.random(shape) < 0.03] = 0.0
    if spoil is not None:
        pick = rng.random(shape) < 0.15
        odf[pick, rng.integers(0, nverts)] = spoil
    p = W.base_params(shape, nverts, nverts, len(edges), step, "PROB")
    p.update(max_sline_len=60, sphere_symm=symm)
    w = W.Workload("prob", p, odf, stop, verts, edges)
    lo, hi = -0.4, np.array(shape) - 0.7
    seeds = (lo + rng.random((48, 3)) * (hi - lo)).astype(np.float32)
    return w, seeds


def _check(w, seeds):
    g, o = _run_both(w, seeds)
    assert len(o["sline_len"]) > 0
    _assert_same(g, o)


@pytest.mark.parametrize("nverts", [66, 254, 258, 362, 510, 514, 724, 768, 770])
def test_sphere_sizes(nverts):
    _check(*_workload(nverts))


@pytest.mark.parametrize("step", [0.05, 0.9, 1.7])
def test_cell_moves(step):
    _check(*_workload(724, step=step))


@pytest.mark.parametrize("shape", [(1, 9, 8), (9, 1, 8), (9, 8, 1), (2, 2, 2)])
def test_thin_volumes(shape):
    _check(*_workload(362, shape=shape))


@pytest.mark.parametrize("shape", [(256, 3, 2), (257, 3, 2), (3, 2, 520)])
def test_long_volumes(shape):
    """Seed-order bricks of 4 voxels up to 256 voxels, coarser past them."""
    _check(*_workload(66, shape=shape))


def test_symmetric_sphere():
    _check(*_workload(362, symm=1))


@pytest.mark.parametrize("spoil", [np.nan, np.inf, -np.inf, 3e30, 1e38, -5.0])
def test_values_off_the_fast_path(spoil):
    """Against the general kernel (per-seed nesting), and against the oracle
    too except with NaN, where the oracle's serial maximum differs from the
    lanes' tree."""
    w, seeds = _workload(362, spoil=np.float32(spoil))
    g, o = _run_both(w, seeds)
    n, _ = _run_both(w, seeds, flat=False)
    assert len(g["sline_len"]) > 0
    for k in ("counts", "sline_seed", "sline_len", "points"):
        assert np.array_equal(g[k], n[k], equal_nan=k == "points"), k
    if not np.isnan(spoil):
        _assert_same(g, o)


def test_negative_and_zero_pmf():
    w, seeds = _workload(362)
    w.dataf[:, :, :6] *= -1.0
    w.dataf[:, :, 6:8] = 0.0
    _check(w, seeds)
