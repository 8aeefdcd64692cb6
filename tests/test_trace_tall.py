"""The tracer on the tallest images: more rows of 8x8 tiles than the second
dimension of a grid holds (65535), up to the 1048560 rows that the entry point
takes.  Pixel for pixel against the oracle's walk."""
import numpy as np
import pytest

from test_trace import camera

DEPTH = 4


def run(m, oracle, heights):
    rng = np.random.default_rng(0x7A11)
    words = oracle.create_final_dag(oracle.create_dag(rng.integers(0, 1 << (3 * DEPTH), size=500, dtype=np.uint64), DEPTH))
    side = float(1 << DEPTH)
    for height in heights:
        print(f"[trace-tall] 1x{height}", flush=True)
        p = camera(DEPTH, (-0.4 * side, -0.3 * side, -0.5 * side), (0.5 * side,) * 3, 1, height)
        want_p, want_c = oracle.trace_paths(words, DEPTH, p)
        got_p, got_c = m.trace_paths(words, DEPTH, p)
        assert np.array_equal(got_p, want_p) and np.array_equal(got_c, want_c)


def test_tall_images_on_the_cpu_emulator(oracle):
    import emu_ctypes
    m = emu_ctypes.use_emulator()
    try:
        run(m, oracle, (8 * 65535 + 1,))
    finally:
        from dag_compression_fast_amd import _lib
        m._default = None
        _lib._lib = None
        _lib._hip = None


@pytest.mark.gpu
def test_tall_images_on_gpu(gpu, oracle):
    run(gpu, oracle, (8 * 32768, 8 * 32768 + 1, 8 * 65535 + 1, 16 * 65535))
