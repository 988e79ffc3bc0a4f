"""bench.py names the kernel that its seeds launch: on both sides of the
bootstrap variants' threshold, pinned or not."""

import os
import sys
import types

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("mode,occ,waves,stepping,want", [
    ("mfma", 0, 2, "flat", "phase2_boot_batch_kernel<1, 2, true>"),
    ("mfma", 0, 4, "flat", "phase2_boot_batch_kernel<1, 4, true>"),
    ("mfma", 4, 2, "flat", "phase2_boot_batch_kernel<1, 4, true>"),
    ("exact", 0, 2, "flat", "phase2_queue_kernel<1, 6>"),
    ("exact", 0, 4, "flat", "phase2_queue_kernel<1, 4>"),
    ("exact", 2, 4, "flat", "phase2_queue_kernel<1, 6>"),
    ("exact", 0, 2, "seed", "phase2_queue_kernel<1, 0>"),
])
def test_bootstrap_variant(mode, occ, waves, stepping, want):
    sys.path.insert(0, ROOT)
    import bench

    args = types.SimpleNamespace(getter="csa", boot_mode=mode, boot_occ=occ, ptt_lanes=0, stepping=stepping)
    assert bench.kernel_name(args, True, waves) == want
