"""Leaf reduce over 64^3 cells (keys grouped by code >> 18 with known cell
starts): plain builds of depths 7 to 9 after one pass, of depths 10 and 11
below a top digit, and batched builds of chunk depths 7 to 9.  Sizes sit at the
edges of the choice (the fewest keys that take it, 16 keys a cell), of a round
of loads (4096 keys of one cell and its neighbours), and of the runs of cells;
empty cells lie first, last and between.  Integer output, equal to the oracle's
bit for bit."""
import numpy as np
import pytest

from dagcheck import assert_dag_equal


def cell_keys(rng, depth, cells, counts):
    """counts[i] random keys in cell cells[i], shuffled."""
    total = 1 << (3 * depth - 18)
    parts = [(np.uint64(c % total) << np.uint64(18)) | rng.integers(0, 1 << 18, size=k, dtype=np.uint64)
             for c, k in zip(cells, counts)]
    keys = np.concatenate(parts)
    return keys[rng.permutation(len(keys))]


def plain(m, oracle, keys, depth, mode=1):
    from dag_compression_fast_amd import _lib
    ctx = m.Context()
    try:
        ctx.set_option(_lib.OPT_TOP_DIGIT_FIRST, mode)
        print(f"[cells] depth {depth} {keys.dtype} {len(keys)} keys mode {mode}", flush=True)
        dag = m.create_dag(keys, depth, ctx=ctx)
        exp = oracle.create_dag(keys, depth)
        assert_dag_equal(dag.to_numpy(), exp, f"depth {depth} {len(keys)} keys")
        assert dag.pre_dedup == exp["pre_dedup"]
        dag.free()
    finally:
        ctx.close()


def batched(m, oracle, chunks, depth):
    keys, offsets = np.concatenate(chunks), np.zeros(len(chunks) + 1, dtype=np.uint64)
    offsets[1:] = np.cumsum([len(c) for c in chunks])
    print(f"[cells] {len(chunks)} chunks of depth {depth}, {len(keys)} keys", flush=True)
    dag = m.create_dag_batched(keys, offsets, depth)
    union = np.concatenate([(np.uint64(i) << np.uint64(3 * depth)) | c for i, c in enumerate(chunks)])
    extra = {1: 0, 8: 1, 64: 2}[len(chunks)]
    assert_dag_equal(dag.to_numpy(), oracle.create_dag(union, depth + extra), f"{len(chunks)} chunks")
    dag.free()


def run_plain(m, oracle):
    rng = np.random.default_rng(0xCE11)
    for depth in (7, 8, 9):
        last = (1 << (3 * depth - 18)) - 1
        for n in (1, 255, 256, 257, 511, 1000):
            keys = rng.integers(0, 1 << (3 * depth), size=n, dtype=np.uint64)
            plain(m, oracle, keys, depth)
            plain(m, oracle, keys.astype(np.uint32), depth)
        keys = cell_keys(rng, depth, [0, 2, last], [4095, 4096, 4097])
        plain(m, oracle, keys, depth)
        plain(m, oracle, keys.astype(np.uint32), depth)
        keys = cell_keys(rng, depth, [1, last - 1, 5, 3], [8193, 511, 512, 513])
        plain(m, oracle, keys, depth)
    # A full cell, every key of one leaf, and the last voxel alone.
    plain(m, oracle, np.arange(3 << 18, (3 << 18) + (1 << 18), dtype=np.uint64)[::-1].copy(), 8)
    plain(m, oracle, np.full(5000, (1 << 27) - 1, dtype=np.uint64), 9)


def run_below_top(m, oracle, sizes):
    rng = np.random.default_rng(0xCE12)
    for depth, n, mode in sizes:
        cells = rng.integers(0, 1 << (3 * depth - 18), size=max(1, n // 700))
        keys = cell_keys(rng, depth, cells, [700] * len(cells))
        plain(m, oracle, keys, depth, mode)


def run_batched(m, oracle):
    rng = np.random.default_rng(0xCE13)
    for depth, num, most in ((7, 8, 3000), (8, 8, 3000), (9, 8, 9000), (7, 64, 800), (9, 1, 20000)):
        last = (1 << (3 * depth - 18)) - 1
        chunks = []
        for i in range(num):
            k = int(rng.integers(1, most))
            cells = [0, last, int(rng.integers(0, last + 1))]
            chunks.append(cell_keys(rng, depth, cells, [k, 1 + k // 3, 1 + k // 2]))
        for i in ((0, num - 1, num // 2) if num > 1 else ()):  # empty chunks, first and last among them
            chunks[i] = chunks[i][:0]
        batched(m, oracle, chunks, depth)
    # Below 16 keys a cell over many cells: the 32^3 groups take it.
    chunks = [rng.integers(0, 1 << 27, size=1500, dtype=np.uint64) for _ in range(64)]
    batched(m, oracle, chunks, 9)


@pytest.fixture(scope="module")
def emu():
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    yield svd
    from dag_compression_fast_amd import _lib
    _lib._lib = None
    _lib._hip = None
    svd._default = None


def test_cells_on_the_cpu_emulator(emu, oracle):
    run_plain(emu, oracle)
    run_below_top(emu, oracle, [(10, 40_000, 2)])
    run_batched(emu, oracle)


@pytest.mark.gpu
def test_cells_on_gpu(gpu, oracle):
    run_plain(gpu, oracle)
    run_below_top(gpu, oracle, [(10, 1_100_000, 1), (11, 1_100_000, 1), (12, 4_300_000, 1), (12, 1_100_000, 1)])
    run_batched(gpu, oracle)


def run_sparse(m, oracle):
    """Batched builds most of whose chunks are empty sort only the others: half
    of the chunks (the most that takes it), one, the first and the last."""
    rng = np.random.default_rng(0xCE14)
    for depth, num, live in ((7, 8, (0, 3, 5, 7)), (9, 64, (63,)), (8, 64, (0, 17, 18, 63)), (9, 8, (2,)),
                             (7, 8, (0, 1, 2, 3, 4))):
        chunks = [np.empty(0, dtype=np.uint64) for _ in range(num)]
        last = (1 << (3 * depth - 18)) - 1
        for i in live:
            chunks[i] = cell_keys(rng, depth, [0, last, last // 2], [700, 1, 4100])
        batched(m, oracle, chunks, depth)


def test_sparse_chunks_on_the_cpu_emulator(emu, oracle):
    run_sparse(emu, oracle)


@pytest.mark.gpu
def test_sparse_chunks_on_gpu(gpu, oracle):
    run_sparse(gpu, oracle)
