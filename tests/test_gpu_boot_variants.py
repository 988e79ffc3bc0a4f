"""Both occupancy variants of the bootstrap kernels, whatever the number of
seeds would choose: the exact kernel at 4 waves per SIMD, which the larger runs
take, bit-exact against the CPU oracle at the matrix sizes where its two
layouts and its blocks can go wrong; at the full volume, where the 2-waves
variants are compared with the oracle and with each other, the 4-waves ones
equal to them."""

import numpy as np
import pytest

from test_gpu_boot_batch import _seeds, _workload
from test_gpu_boot_mfma import _track

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("occ", [2, 4])
@pytest.mark.parametrize("kind,dirs,order,verts", [
    ("csa", 16, 2, 362), ("csa", 17, 2, 66), ("csa", 32, 4, 362), ("csa", 33, 4, 64), ("opdt", 31, 4, 362),
    ("opdt", 36, 4, 362), ("opdt", 100, 6, 724), ("csa", 101, 6, 362), ("csa", 100, 8, 724), ("csa", 160, 6, 724)])
def test_exact_variant_against_the_oracle(kind, dirs, order, verts, occ):
    from conftest import packed_points
    from oracle.oracle import Oracle

    w = _workload(kind, dirs, order, verts)
    seeds = _seeds(w, 9)
    g = _track(w, seeds, 0, occ=occ)
    o = Oracle(w.params, w.dataf, w.stop_map, w.vertices, w.edges, boot=w.boot).track(seeds)
    assert len(o["sline_len"]) > 0
    for k in ("counts", "sline_seed", "sline_len"):
        assert np.array_equal(g[k], o[k]), k
    assert np.array_equal(g["points"], packed_points(o))


@pytest.mark.parametrize("mode,n", [(0, 8000), (1, 20000)])
@pytest.mark.parametrize("kind", ["csa", "opdt"])
def test_variants_agree_at_the_full_volume(kind, mode, n):
    from gpustreamlines_amd import workloads as W

    w = W.build(kind)
    seeds = W.seeds_for(w, n, placement="mask", seed=1)
    print(f"[boot-variants] {kind} mode={mode} 81x106x76 seeds={n}", flush=True)
    a, b = (_track(w, seeds, mode, rng_chunk=25000, occ=occ) for occ in (2, 4))
    assert len(a["sline_len"]) > n
    for k in ("counts", "sline_seed", "sline_len", "points"):
        assert np.array_equal(a[k], b[k]), k
