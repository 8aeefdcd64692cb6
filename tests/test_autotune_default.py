"""The time that the autotuner reports for the defaults is that of a fresh
context's options, which leave the segmented sort's first digit to the library
(0), not of the two-pass split that digit 0 once stood for."""
from test_autotune import FakeCtx, setting_of

import numpy as np
import pytest

from dag_compression_fast_amd import autotune


def cost(setting):
    return 1.0 + 0.25 * setting["seg_first_bits"] + 0.125 * setting["table_load_shift"]


def tune(space):
    ctx, now = FakeCtx(), [0.0]

    def build(c):
        now[0] += cost(setting_of(c)) / 1e3

    return autotune.autotune(ctx, build, lambda: np.arange(4, dtype=np.uint32), reps=1, space=space,
                             clock=lambda: now[0], chunk_depth=9)


def test_default_time_is_the_librarys_choice():
    res = tune(autotune.SEG_SPACE)
    fresh = {"seg_first_bits": 0, "table_load_shift": 1}
    assert autotune.library_setting(autotune.SEG_SPACE) == fresh
    assert res["default_ms"] == pytest.approx(cost(fresh))
    assert res["default_ms"] != pytest.approx(cost({"seg_first_bits": 6, "table_load_shift": 1}))


def test_no_default_time_without_the_default():
    assert tune({"seg_first_bits": (4, 6), "table_load_shift": (1, 2)})["default_ms"] is None
