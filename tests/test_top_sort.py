"""svdag_sort_keys top digit first (64-bit keys, three digits or more, at most 32
bits below the top one), against numpy: random keys, all in one bucket, few
values, sizes around a tile (4096) and the smallest that takes it by itself,
the widest and narrowest spans, and keys with higher bits (kept by the LSD
sort, which must take over).  Equal keys are identical, so the sorted keys are
unique: integer output, tolerance 0."""
import numpy as np
import pytest

ALWAYS = 2


def check(m, keys, bits, what, radix=None, mode=None):
    from dag_compression_fast_amd import _lib
    ctx = m.Context()
    try:
        if radix:
            ctx.set_option(_lib.OPT_RADIX_BITS, radix)
        if mode is not None:
            ctx.set_option(_lib.OPT_TOP_DIGIT_FIRST, mode)
        print(f"[top-sort] {what}: {len(keys)} keys, {bits} bits", flush=True)
        got = m.sort_keys(keys, bits, ctx=ctx)
        low = keys & np.uint64((1 << bits) - 1)
        assert np.array_equal(got, keys[np.argsort(low, kind="stable")]), what
    finally:
        ctx.close()


def inputs(rng, n, bits):
    keys = rng.integers(0, 1 << bits, size=n, dtype=np.uint64)
    yield "random", keys
    yield "one bucket", keys >> np.uint64(10)
    yield "three values", rng.choice(np.array([0, 5, (1 << bits) - 1], dtype=np.uint64), size=n)
    yield "ends", np.where(rng.random(n) < 0.5, keys, np.uint64((1 << bits) - 1))
    wide = keys.copy()
    wide[n // 2] |= np.uint64(1) << np.uint64(bits)
    yield "one higher bit", wide


def test_top_sort_on_the_cpu_emulator():
    import emu_ctypes
    m = emu_ctypes.use_emulator()
    try:
        rng = np.random.default_rng(0x705)
        for n, bits, radix in ((12288, 13, 4), (8191, 12, 4), (20001, 36, 5), (16385, 20, 5)):
            for what, keys in inputs(rng, n, bits):
                check(m, keys, bits, what, radix, ALWAYS)
    finally:
        from dag_compression_fast_amd import _lib
        import dag_compression_fast_amd as svd
        _lib._lib = None
        _lib._hip = None
        svd._default = None


@pytest.mark.gpu
def test_top_sort_on_gpu(gpu):
    rng = np.random.default_rng(0x706)
    for n, bits in (((1 << 22) - 1, 33), (1 << 22, 33), ((1 << 22) + 1, 41), (5_000_003, 19), (6_000_000, 42),
                    (20_000_001, 27)):
        for what, keys in inputs(rng, n, bits):
            check(gpu, keys, bits, what)
    for what, keys in inputs(rng, 300_001, 24):
        check(gpu, keys, 24, what, 4, ALWAYS)
