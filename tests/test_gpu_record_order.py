"""Recorded training pairs are a sample of the seeds whatever their number of
directions: a buffer that fills up must not hold those of the seeds with the
most directions only (the order in which a plain run takes its seeds).  A
seed's random stream follows its index, so the pairs of the seeds with few
directions are known exactly from a run of those alone, put first."""

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_full_buffer_holds_pairs_of_seeds_of_all_direction_counts(small_workloads):
    from gpustreamlines_amd import learned as LP
    from gpustreamlines_amd import workloads as W
    from gpustreamlines_amd._device import DeviceTracker

    w0 = small_workloads["ptt"]
    w = dataclasses.replace(w0, params=dict(w0.params, max_sline_len=16))
    seeds = W.seeds_for(w, 8000, placement="mask", seed=3)
    dt = DeviceTracker(w.params, device=0)
    try:
        dt.upload(w.dataf, w.stop_map, w.vertices, w.edges, ptt_lut=w.ptt_lut)
        dt.set_launch(0, 64, 1)  # 512 slots on 256 CUs: most seeds wait in the queue
        counts = dt.track(seeds)["counts"]
        seeds, counts = seeds[counts > 0], counts[counts > 0]
        by = np.argsort(counts, kind="stable")
        seeds, counts = seeds[by], counts[by]
        few = int(np.searchsorted(counts, np.median(counts), side="right"))
        print(f"[record] {len(seeds)} seeds, {few} of at most {counts[few - 1]} directions, "
              f"{np.bincount(counts)}", flush=True)
        assert 0 < few < len(seeds)

        def record(s, capacity):
            buf, n = LP.record_pairs(dt, s, capacity, 0.02, rng_chunk=len(seeds))
            try:
                return buf.download(np.zeros((n, LP.PAIR), np.float32))
            finally:
                buf.free()

        part = record(seeds[:few], 2_000_000)
        full = record(seeds, 2_000_000)
        assert 1000 < len(part) < len(full) < 2_000_000
        rows = {r.tobytes() for r in part}
        share = sum(r.tobytes() in rows for r in full) / len(full)
        assert abs(share - len(part) / len(full)) < 1e-3  # the same streams in both runs
        first = record(seeds, len(full) // 4)
        assert len(first) == len(full) // 4
        kept = sum(r.tobytes() in rows for r in first) / len(first)
        print(f"[record] share of the pairs {share:.3f}, of a quarter's buffer {kept:.3f}", flush=True)
        # a uniform sample would hold `share`; the queue's first seeds are another region, not another kind
        assert kept > share / 2
    finally:
        dt.close()
