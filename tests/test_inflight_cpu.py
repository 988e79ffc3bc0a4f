"""One chunk per launch: as many handles as there are chunks, up to the
pipeline's depth (a handle of the family counts as having seeds in flight)."""

import numpy as np
import pytest

from gpustreamlines_amd import propagate_seeds
from gpustreamlines_amd.generic_tracker import GenericTracker


@pytest.mark.parametrize("nseeds,launch_seeds,want", [(200, 0, 8), (30, 0, 3), (15, 0, 2), (100, 20, 2)])
def test_pipeline_depth(monkeypatch, nseeds, launch_seeds, want):
    depths = []

    class Pipe:
        def __init__(self, dt, depth, **kw):
            depths.append(depth)

        def run(self, seeds, step, sink=None):
            for c in range(0, len(seeds), step):
                yield np.zeros((0, 3), np.float32), np.zeros(0, np.int64)

        def close(self):
            pass

    class Tracker(GenericTracker):
        chunk_size, chunk_pipeline = 10, 8
        device_trackers = [None]
        seed_propagator = None

    monkeypatch.setattr(propagate_seeds, "ChunkPipeline", Pipe)
    t = Tracker()
    t.launch_seeds = launch_seeds
    assert sum(n for _, _, n in t._raw_chunks(np.zeros((nseeds, 3), np.float32))) == nseeds
    assert depths == [want]
