"""The exact bootstrap kernel's products at the matrix sizes where their
blocks of 32 rows and columns can go wrong, bit-exact against the CPU oracle:
columns a multiple of 4 or not (the two layouts), of 32 or not, fewer than a
block, and spheres whose rows end inside one."""

import pytest

from test_gpu_boot_batch import _seeds, _workload
from test_gpu_parity import _assert_same, _run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,dirs,order,verts", [
    ("csa", 16, 2, 362), ("csa", 17, 2, 66), ("csa", 32, 4, 362), ("csa", 33, 4, 64), ("opdt", 31, 4, 362),
    ("opdt", 36, 4, 362), ("csa", 101, 6, 362), ("csa", 100, 8, 724)])
def test_sizes(kind, dirs, order, verts):
    w = _workload(kind, dirs, order, verts)
    g, o = _run_both(w, _seeds(w, 9))
    assert len(o["sline_len"]) > 0
    _assert_same(g, o)


def test_large_run_has_the_small_runs_prefix():
    """More than 8 seeds a slot (32,768 on 256 CUs) take the variant of 4 waves per SIMD."""
    import numpy as np
    from test_gpu_boot_mfma import _track

    w = _workload("csa", 33, 4, 64)
    seeds = _seeds(w, 33000)
    full = _track(w, seeds, 0)
    part = _track(w, seeds[:500], 0)
    k, pts = len(part["sline_len"]), int(part["point_offsets"][-1])
    assert k > 0 and np.array_equal(part["counts"], full["counts"][:500])
    assert np.array_equal(part["sline_len"], full["sline_len"][:k])
    assert np.array_equal(part["points"], full["points"][:pts])
