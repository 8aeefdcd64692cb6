"""svdag_sort_keys top digit first on keys with bits above the sorted ones: such
keys keep those bits and, equal on the sorted ones, their order.  Even and odd
numbers of passes below the top digit, a few values (long runs of equal low
bits, so that any change of order shows), an output that starts inside the
input, and one histogram for either kind of key.  Integer output, tolerance 0
against numpy's stable sort."""
import numpy as np
import pytest

ALWAYS = 2


def inputs(rng, n, bits):
    low = rng.integers(0, 1 << bits, size=n, dtype=np.uint64)
    high = np.arange(n, dtype=np.uint64) << np.uint64(bits)  # every key another, in input order
    yield "all wide", low | high
    yield "wide, few values", rng.choice(low[:5], size=n) | high
    yield "wide, one bucket", (low & np.uint64(255)) | high
    some = low.copy()
    some[rng.integers(0, n, size=max(1, n // 100))] |= np.uint64(1) << np.uint64(63)
    yield "some wide", some


def expected(keys, bits):
    return keys[np.argsort(keys & np.uint64((1 << bits) - 1), kind="stable")]


def run(m, rng, sizes):
    from dag_compression_fast_amd import _lib
    for n, bits, radix, mode in sizes:
        ctx = m.Context()
        try:
            ctx.set_option(_lib.OPT_RADIX_BITS, radix)
            ctx.set_option(_lib.OPT_TOP_DIGIT_FIRST, mode)
            for what, keys in inputs(rng, n, bits):
                print(f"[top-sort-wide] {what}: {n} keys, {bits} bits, digits of {radix}", flush=True)
                assert np.array_equal(m.sort_keys(keys, bits, ctx=ctx), expected(keys, bits)), (what, n, bits)
        finally:
            ctx.close()


def run_overlapping(m, rng, n, bits, radix, mode):
    """The output starts in the middle of the input."""
    from dag_compression_fast_amd import _lib
    keys = rng.integers(0, 1 << 62, size=n, dtype=np.uint64)
    ctx = m.Context()
    try:
        ctx.set_option(_lib.OPT_RADIX_BITS, radix)
        ctx.set_option(_lib.OPT_TOP_DIGIT_FIRST, mode)
        room = m.DeviceBuffer.from_numpy(np.concatenate([keys, np.zeros(n, dtype=np.uint64)]))
        at = n // 2
        _lib.check(_lib.lib().svdag_sort_keys(ctx.handle, room.address, n, bits, room.address + 8 * at))
        assert np.array_equal(room.to_numpy(np.uint64, n, 8 * at), expected(keys, bits))
        room.free()
    finally:
        ctx.close()


@pytest.fixture(scope="module")
def emu():
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    yield svd
    from dag_compression_fast_amd import _lib
    svd._default = None
    _lib._lib = None
    _lib._hip = None


def test_wide_keys_on_the_cpu_emulator(emu):
    rng = np.random.default_rng(0x71DE)
    run(emu, rng, [(12288, 12, 4, ALWAYS), (12289, 13, 4, ALWAYS), (20001, 36, 5, ALWAYS), (9000, 17, 4, ALWAYS)])
    run_overlapping(emu, rng, 9001, 12, 4, ALWAYS)
    run_overlapping(emu, rng, 9001, 13, 4, ALWAYS)


def test_one_histogram_for_either_kind_of_key(emu):
    from dag_compression_fast_amd import _lib
    rng = np.random.default_rng(0x71DF)
    low = rng.integers(0, 1 << 12, size=9000, dtype=np.uint64)
    ctx = emu.Context()
    try:
        ctx.set_option(_lib.OPT_RADIX_BITS, 4)
        ctx.set_option(_lib.OPT_TOP_DIGIT_FIRST, ALWAYS)
        for keys in (low, low | np.uint64(1) << np.uint64(40)):
            ctx.profile_enable(["sort_histogram"])
            ctx.profile_reset()
            emu.sort_keys(keys, 12, ctx=ctx)
            assert ctx.profile_read()["sort_histogram"][1] == 1
    finally:
        ctx.close()


@pytest.mark.gpu
def test_wide_keys_on_gpu(gpu):
    rng = np.random.default_rng(0x71E0)
    run(gpu, rng, [(300_001, 24, 4, ALWAYS), (1 << 22, 27, 9, ALWAYS), (8_400_001, 33, 9, 1), (8_388_608, 41, 9, 1)])
    run(gpu, rng, [(36_000_003, 19, 9, 1)])  # slices of several tiles
    run_overlapping(gpu, rng, 8_500_000, 27, 9, 1)
