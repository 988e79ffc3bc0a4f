"""The autotuner's choice without a GPU: the library's own setting is timed for
every getter, wins when it is within the noise of the best, and tuning the
bootstrap kernel keeps the mode's flags."""

import pytest

from gpustreamlines_amd import autotune


@pytest.mark.parametrize("model,mode", [(0, 0), (1, 0), (0, 1), (1, 1), (2, 0), (3, 0)])
def test_library_default_is_a_candidate(model, mode):
    c = list(autotune.candidates(model, mode))
    d = autotune.default(model, mode)
    assert c[0] == d
    assert d["threads"] == d["blocks_per_cu"] == d["lanes"] == d["schedule"] == 0 and d["flat"]
    assert ("waves_per_simd" in d) == (mode == 1) and not d.get("waves_per_simd")
    keys = [tuple(sorted(x.items())) for x in c]
    assert len(set(keys)) == len(keys)


def test_default_wins_within_the_margin():
    assert autotune.pick({"auto": 104.0, "a": 100.0, "b": 200.0}, "auto") == "auto"
    assert autotune.pick({"auto": 106.0, "a": 100.0, "b": 200.0}, "auto") == "a"
    assert autotune.pick({"auto": 90.0, "a": 100.0}, "auto") == "auto"


@pytest.mark.parametrize("full", [False, True])
def test_apply_keeps_the_product_form(full):
    class Dt:
        BOOT_MFMA = 1
        params = dict(model_type=1)
        boot_full = full

        def set_launch(self, *a):
            pass

        set_stepping = set_launch

        def set_boot_mode(self, *a):
            self.got = a

    dt = Dt()
    autotune.apply(dt, autotune.default(1, 1))
    assert dt.got == (1, 0, full)
