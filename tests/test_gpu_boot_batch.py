"""The batched bootstrap kernel at the sizes where its tiles, rows and slots can
go wrong: signal lengths around the 16-row tiles and 32-lane rows, spheres
below and above one block of 512 vertices, no adjacency table, a NaN in the
signal.  Its two occupancy variants do the same operations in the same order
and must agree exactly; against the exact kernel the bar is the batched
kernel's: the same streamlines, most of them bit-identical.  A seed's result
depends on nothing but its index, so any number of seeds gives the prefix of a
larger run."""

import dataclasses
import functools

import numpy as np
import pytest

from test_gpu_boot_mfma import _track

pytestmark = pytest.mark.gpu

SHAPE = (20, 22, 18)


@functools.lru_cache(maxsize=8)
def _workload(kind, dirs, order, verts):
    from gpustreamlines_amd import workloads as W
    from gpustreamlines_amd.boot_utils import prepare_csa, prepare_opdt
    from gpustreamlines_amd.phantom import make_phantom
    from gpustreamlines_amd.sphere import single_shell_gtab, symmetric_sphere

    ph = make_phantom(SHAPE, gtab=single_shell_gtab(3, dirs), seed=3)
    sv, edges = symmetric_sphere(verts)
    prep = (prepare_csa if kind == "csa" else prepare_opdt)(ph.gtab, sv, sh_order_max=order)
    boot = {k: np.ascontiguousarray(prep[k], dtype=np.float32)
            for k in ("H", "R", "delta_b", "delta_q", "sampling_matrix")}
    boot["b0s_mask"] = np.asarray(prep["b0s_mask"], dtype=np.int32)
    p = W.base_params(SHAPE, ph.dwi.shape[3], len(sv), len(edges), 0.5, kind.upper())
    p["delta_nr"] = boot["delta_b"].shape[0]
    return W.Workload(kind, p, ph.dwi, ph.fa, sv, edges, boot=boot, extra=dict(phantom=ph))


def _seeds(w, n):
    from gpustreamlines_amd import workloads as W

    return W.seeds_for(w, n, placement="mask", seed=5)


def _same(a, b):
    for k in ("counts", "sline_seed", "sline_len", "points"):
        assert np.array_equal(a[k], b[k], equal_nan=k == "points"), k


def _check(w, n=150, full=False):
    seeds = _seeds(w, n)
    a = _track(w, seeds, 1, occ=2, full=full)
    _same(a, _track(w, seeds, 1, occ=4, full=full))
    b = _track(w, seeds, 0)
    assert np.array_equal(a["counts"], b["counts"]) and np.array_equal(a["sline_seed"], b["sline_seed"])
    assert len(a["sline_len"]) > 0
    pa, pb = a["point_offsets"], b["point_offsets"]
    same = np.mean([np.array_equal(a["points"][pa[i]:pa[i + 1]], b["points"][pb[i]:pb[i + 1]])
                    for i in range(len(a["sline_len"]))])
    print(f"identical {same:.4f} of {len(a['sline_len'])}", flush=True)
    assert same >= 0.7


@pytest.mark.parametrize("kind,dirs,order,verts", [
    ("csa", 16, 2, 362), ("csa", 17, 2, 66), ("csa", 33, 4, 362), ("opdt", 31, 4, 512), ("opdt", 65, 6, 514),
    ("csa", 101, 6, 768), ("csa", 270, 8, 724), ("opdt", 270, 8, 362)])
def test_sizes(kind, dirs, order, verts):
    _check(_workload(kind, dirs, order, verts))


def test_full_products():
    _check(_workload("csa", 101, 6, 768), full=True)


def test_no_adjacency_table():
    """A vertex of more than 8 neighbours: the edge form of the peak search."""
    w = _workload("csa", 33, 4, 362)
    ends = {int(x) for e in w.edges for x in e if 0 in e}
    extra = [(0, v) for v in range(100, 110) if v not in ends]
    edges = np.concatenate([w.edges, np.asarray(extra, dtype=w.edges.dtype)])
    _check(dataclasses.replace(w, edges=edges, params=dict(w.params, nedges=len(edges))))


def test_nan_signal():
    w = _workload("csa", 33, 4, 362)
    data = w.dataf.copy()
    data[8:10, 9:11, 8, 20] = np.nan
    _check(dataclasses.replace(w, dataf=data))


@pytest.mark.parametrize("n", [1, 2, 17, 255, 257, 600])
def test_few_seeds_are_a_prefix(n):
    w = _workload("csa", 33, 4, 362)
    seeds = _seeds(w, 5000)
    full = _track(w, seeds, 1, occ=4)
    part = _track(w, seeds[:n], 1)
    k = len(part["sline_len"])
    pts = int(part["point_offsets"][-1])
    assert np.array_equal(part["counts"], full["counts"][:n])
    assert np.array_equal(part["sline_len"], full["sline_len"][:k])
    assert np.array_equal(part["points"], full["points"][:pts])
