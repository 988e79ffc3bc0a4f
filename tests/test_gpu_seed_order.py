"""The workspace of a bounded chunk: what callers were told to allocate when
the seed order had one bucket per 4-voxel brick (volumes of up to 512 voxels a
side) stays enough, whatever the order's classes need on top."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _one_bucket_per_brick(dims, n, cap):
    """Bytes of that workspace: order, keys, counts, starts and block sums,
    then the block sums of the two scans, aligned to 256."""
    mx, log2 = max(dims), 2
    while (mx - 1) >> log2 >= 128:
        log2 += 1
    nb = 1 << (3 * ((mx - 1) >> log2).bit_length())

    def up(x):
        return -(-x // 256) * 256

    return up(4 * (2 * n + 2 * nb + 1 + -(-nb // 1024))) + up(4 * -(-n // 1024)) + 8 * -(-cap // 1024)


@pytest.mark.parametrize("dims", [(3, 2, 4), (13, 11, 12), (81, 106, 76), (257, 9, 8), (600, 3, 2)])
@pytest.mark.parametrize("n,cap", [(1, 1), (1025, 3000), (25000, 200000)])
def test_workspace_does_not_grow(dims, n, cap):
    from gpustreamlines_amd import _lib
    from gpustreamlines_amd import workloads as W
    from gpustreamlines_amd._device import DeviceTracker

    dt = DeviceTracker(W.base_params(dims, 66, 66, 100, 0.5, "PROB"))
    try:
        b = C.c_size_t()
        _lib.check(dt.L.cuslines_chunk_workspace_bytes(dt.h, n, cap, C.byref(b)), "chunk_workspace")
    finally:
        dt.close()
    assert 8 * n <= b.value <= _one_bucket_per_brick(dims, n, cap)


@pytest.mark.parametrize("kind", ["prob", "ptt", "csa"])
def test_chunk_runs_in_that_workspace(small_workloads, kind):
    from gpustreamlines_amd import workloads as W
    from gpustreamlines_amd._device import ChunkBuffers, DeviceTracker

    w = small_workloads[kind]
    seeds = W.seeds_for(w, 200, placement="mixed", seed=6)
    dt = DeviceTracker(w.params, device=0)
    try:
        dt.upload(w.dataf, w.stop_map, w.vertices, w.edges, boot=w.boot, ptt_lut=w.ptt_lut)
        ref = dt.track(seeds)
        cb = ChunkBuffers(dt, len(seeds), 20 * len(seeds))
        try:
            dims = tuple(w.params[k] for k in ("dimx", "dimy", "dimz"))
            need = _one_bucket_per_brick(dims, len(seeds), cb.cap)
            whole = cb._alloc(need + 256)
            whole.upload(np.full(need // 4 + 64, 77, np.int32))
            cb.ws = whole.part(0, need)
            cb.sd.upload(seeds)
            cb.enqueue(len(seeds), len(seeds))
            got = cb.collect(len(seeds))
            assert (whole.download(np.zeros(need // 4 + 64, np.int32))[need // 4:] == 77).all()
        finally:
            cb.close()
    finally:
        dt.close()
    assert got["totals"][0] == got["totals"][1] == len(ref["sline_len"]) > 0
    assert np.array_equal(got["sline_len"], ref["sline_len"]) and np.array_equal(got["points"], ref["points"])
