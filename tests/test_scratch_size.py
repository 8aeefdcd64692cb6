"""Scratch of small calls (a context's arena after one call, so also the
smallest memory budget that accepts it): no more than these calls took when the
leaf order was a radix sort and the compactions had scan launches.  On the CPU
emulator, whose plans are the library's."""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def emu():
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    yield svd
    from dag_compression_fast_amd import _lib
    svd._default = None
    _lib._lib = None
    _lib._hip = None


def keys_of(n, depth, salt=0):
    """n keys spread over the grid, no two in one leaf while it has as many."""
    step = max(64, (1 << (3 * depth)) // n)
    return (np.arange(n, dtype=np.uint64) * np.uint64(step) + np.uint64(salt % 64)) & np.uint64((1 << (3 * depth)) - 1)


def scratch_of(svd, call):
    ctx = svd.Context()
    try:
        keep = call(ctx)
        used = ctx.memory_usage()["scratch"]
        for k in keep:
            k.close() if hasattr(k, "close") else k.free()
        return used
    finally:
        ctx.close()


# (depth, keys): bytes
BUILDS = {
    (3, 1): 127488, (3, 24000): 998912, (4, 300): 133120, (6, 1000): 237824, (8, 1): 278528, (8, 1000): 555776,
    (8, 4096): 1451520, (8, 4097): 1754624, (8, 6000): 2044928, (11, 1000): 918272, (11, 5000): 3281664,
    (14, 3000): 2911744,
}
# (depth, keys a DAG, levels): bytes
MERGES = {
    (4, 1, 0): 186112, (4, 20, 2): 306176, (6, 1, 1): 188160, (6, 500, 1): 301568, (6, 500, 2): 1221120,
    (8, 1, 0): 186368, (8, 20, 2): 466176, (8, 3000, 0): 236544, (8, 4500, 0): 205824, (8, 3000, 1): 663296,
}
# (chunk depth, slot levels, keys, max_nodes): bytes
RESIDENTS = {
    (4, 1, 1, 10): 134656, (6, 1, 300, 3000): 242688, (9, 4, 1, 10): 189440, (9, 4, 5000, 50000): 1962752,
    (12, 2, 1, 10): 134912, (12, 2, 1, 100000): 3684096, (12, 2, 300, 3000): 242432, (12, 2, 5000, 50000): 1908480,
    (18, 1, 1, 100000): 3683840, (18, 1, 5, 600000): 28553216,
}


@pytest.mark.parametrize("shape", BUILDS)
def test_builds(emu, shape):
    depth, n = shape
    assert scratch_of(emu, lambda ctx: [emu.create_dag(keys_of(n, depth), depth, ctx=ctx)]) <= BUILDS[shape]


@pytest.mark.parametrize("shape", MERGES)
def test_merges(emu, shape):
    depth, n, k = shape
    dags = [emu.create_dag(keys_of(n, depth, i), depth) for i in range(8 ** k)]
    assert scratch_of(emu, lambda ctx: [emu.merge_dags(dags, ctx=ctx)]) <= MERGES[shape]


@pytest.mark.parametrize("shape", RESIDENTS)
def test_residents(emu, shape):
    depth, top, n, most = shape
    offsets = np.full(8 ** top + 1, n, dtype=np.uint64)
    offsets[0] = 0
    one = emu.create_dag_batched(keys_of(n, depth), offsets, depth)

    def call(ctx):
        r = emu.ResidentDag(depth, top, most, ctx=ctx)
        r.insert(one)
        return [r.dag(), r]

    assert scratch_of(emu, call) <= RESIDENTS[shape]
