"""The voxelizer under a memory budget: what fitted when the columns were tested
twice without anything stored between the passes still fits (the write pass
then makes the tests again), and gives the same keys in the same order as
without a budget.  A byte less than the rows and keys need is still refused."""
import numpy as np
import pytest

# (triangles, depth, edge): the smallest budget of that kind
BUDGETS = {
    (1, 9, 200): 77312, (12, 8, 60): 321792, (60, 8, 60): 2267648, (400, 10, 3): 287488, (3000, 10, 3): 2163712,
    (60, 9, 100): 5528320,
}


def soup(count, depth, edge):
    rng = np.random.default_rng([count, depth, int(10 * edge)])
    return rng.uniform(0, 1 << depth, size=(count, 1, 3)) + rng.normal(0, edge, size=(count, 3, 3))


def keys_under(m, tris, depth, budget):
    from dag_compression_fast_amd import _lib
    ctx = m.Context()
    try:
        ctx.set_option(_lib.OPT_MEMORY_BUDGET, budget)
        buf, n = m.voxelize_triangles(tris, depth, ctx=ctx)
        keys = buf.to_numpy(np.uint64, n)
        buf.free()
        return keys
    finally:
        ctx.close()


def run(m):
    for (count, depth, edge), budget in BUDGETS.items():
        tris = soup(count, depth, edge)
        want = keys_under(m, tris, depth, 0)
        print(f"[voxel-budget] {count} triangles, {len(want)} keys, {budget} bytes", flush=True)
        assert np.array_equal(keys_under(m, tris, depth, budget), want)
        with pytest.raises(m.SvdagError):
            keys_under(m, tris, depth, 8 * len(want))


def test_budget_on_the_cpu_emulator():
    import emu_ctypes
    m = emu_ctypes.use_emulator()
    try:
        run(m)
    finally:
        from dag_compression_fast_amd import _lib
        m._default = None
        _lib._lib = None
        _lib._hip = None


@pytest.mark.gpu
def test_budget_on_gpu(gpu):
    run(gpu)
