"""The completion deadline of a call (SVDAG_OPT_WAIT_SECONDS) holds on every
route of the batched build: a stalled stream fails the call with the stage it
stalled in, and nothing on the way out waits for that stream without a bound.
On the CPU emulator, whose streams report their work unfinished on request."""
import ctypes

import numpy as np
import pytest


@pytest.fixture
def emu():
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    lib = ctypes.CDLL(emu_ctypes.EMU_LIB)
    lib.emu_stream_waits.restype = ctypes.c_uint64
    yield svd, lib
    lib.emu_set_stalled(0)
    from dag_compression_fast_amd import _lib
    svd._default = None  # the emulator's context goes before its library
    _lib._lib = None
    _lib._hip = None


@pytest.mark.parametrize("live", [2, 8])  # chunks with keys of 8: only those sorted, all sorted
def test_a_stalled_batched_build_ends_at_its_deadline(emu, live):
    svd, lib = emu
    from dag_compression_fast_amd import _lib
    rng = np.random.default_rng(17)
    offsets = np.minimum(np.arange(9, dtype=np.uint64), np.uint64(live)) * np.uint64(500)
    keys = svd.DeviceBuffer.from_numpy(rng.integers(0, 1 << 21, size=500 * live, dtype=np.uint64))
    ctx = svd.Context()
    try:
        ctx.set_option(_lib.OPT_WAIT_SECONDS, 1)
        svd.create_dag_batched(keys, offsets, 7, ctx=ctx).free()  # scratch and result blocks are there
        waits = lib.emu_stream_waits()
        lib.emu_set_stalled(1)
        with pytest.raises(svd.SvdagError, match="did not complete within 1 s"):
            svd.create_dag_batched(keys, offsets, 7, ctx=ctx)
        assert lib.emu_stream_waits() == waits, "an unbounded wait for the stalled stream"
        lib.emu_set_stalled(0)
        svd.create_dag_batched(keys, offsets, 7, ctx=ctx).free()
    finally:
        lib.emu_set_stalled(0)
        ctx.close()
