"""Tracer stacks sized by the depth: the depths at which the size changes (9,
12, 16, 21 levels) and their neighbours, image sizes off the 8x8 tiles, against
the oracle's walk, pixel for pixel."""
import numpy as np
import pytest

from test_trace import ALL_ONES, camera

DEPTHS = (3, 8, 9, 10, 12, 13, 16, 17, 20, 21)


def run(m, oracle):
    rng = np.random.default_rng(0x7D)
    for depth in DEPTHS:
        # Clusters of voxels around a few points, so that rays meet some.
        bits = 3 * depth
        seeds = rng.integers(0, 1 << bits, size=40, dtype=np.uint64) & ~np.uint64((1 << max(0, bits - 6)) - 1)
        keys = (seeds[:, None] + rng.integers(0, 1 << max(1, bits - 6), size=(40, 30), dtype=np.uint64)).ravel()
        keys &= np.uint64((1 << bits) - 1)
        words = oracle.create_final_dag(oracle.create_dag(keys, depth))
        side = float(1 << depth)
        for (w, h), dbg in (((33, 17), 0), ((8, 9), ALL_ONES)):
            p = camera(depth, (-0.4 * side, -0.3 * side, -0.5 * side), (0.5 * side,) * 3, w, h, debug_level=dbg)
            want_p, want_c = oracle.trace_paths(words, depth, p)
            got_p, got_c = m.trace_paths(words, depth, p)
            print(f"[trace] depth {depth} {w}x{h}", flush=True)
            assert np.array_equal(got_p, want_p) and np.array_equal(got_c, want_c)


def test_trace_depths_on_the_cpu_emulator(oracle):
    import emu_ctypes
    m = emu_ctypes.use_emulator()
    try:
        run(m, oracle)
    finally:
        from dag_compression_fast_amd import _lib
        import dag_compression_fast_amd as svd
        _lib._lib = None
        _lib._hip = None
        svd._default = None


@pytest.mark.gpu
def test_trace_depths_on_gpu(gpu, oracle):
    run(gpu, oracle)
