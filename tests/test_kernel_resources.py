"""Registers of the built phase-2 kernels, from the code object's own metadata
(no GPU needed): the kernels whose loops were laid out for a register budget
must not spill into scratch memory beyond what their variant was measured
with.  25,000 CSA seeds on the exact kernel's 4-waves variant took 243 ms at
140 spilled vector registers and 230 ms at 74."""

import os
import re
import struct
import subprocess
import tempfile

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def _spills():
    """{mangled kernel name: vgpr_spill_count} of libcuslines_hip.so."""
    from gpustreamlines_amd import _lib

    blob = open(_lib.LIB_PATH, "rb").read()
    at = blob.index(b"__CLANG_OFFLOAD_BUNDLE__")
    (count,) = struct.unpack_from("<Q", blob, at + 24)
    pos = at + 32
    for _ in range(count):
        off, size, n = struct.unpack_from("<QQQ", blob, pos)
        name = blob[pos + 24:pos + 24 + n]
        pos += 24 + n
        if b"gfx950" in name:
            break
    else:
        raise AssertionError("no gfx950 code object")
    with tempfile.NamedTemporaryFile(suffix=".co") as f:
        f.write(blob[at + off:at + off + size])
        f.flush()
        txt = subprocess.run([READELF, "--notes", f.name], capture_output=True, text=True, check=True).stdout
    names = re.findall(r"\.name: +(_Z\w+)\n", txt)
    spills = re.findall(r"\.vgpr_spill_count: +(\d+)", txt)
    assert len(names) == len(spills) > 0
    return dict(zip(names, map(int, spills)))


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_phase2_kernels_spill_no_more_than_measured():
    spills = _spills()

    def worst(pattern):
        got = [v for k, v in spills.items() if re.search(pattern, k)]
        assert got, pattern
        return max(got)

    assert worst(r"phase2_queue_kernelILi[01]ELi[46]E") <= 100  # exact bootstrap, flat stepping
    assert worst(r"phase2_ptt_kernel") == 0
    assert worst(r"phase2_prob_kernel") == 0
    assert worst(r"phase2_boot_batch_kernelILi[01]ELi2E") == 0
    assert worst(r"phase2_boot_batch_kernelILi[01]ELi4E") <= 48
