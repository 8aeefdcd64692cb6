"""Ascending order of the unique leaves (the sample sort of the leaf table's
occupied slots) at the sizes where its buckets change: one bucket, two, many,
and buckets too large for one LDS sort.  The masks come out as np.unique's of
the same masks, and every leaf's parent points at it (decoded words)."""
import numpy as np
import pytest

from dagcheck import assert_dag_equal


def masked_leaves(rng, count, bits):
    """`count` leaves at consecutive codes, each with `bits` random voxels (may
    repeat), as (shuffled keys, unique masks)."""
    low = rng.integers(0, 64, size=(count, bits), dtype=np.uint64)
    keys = ((np.arange(count, dtype=np.uint64) << np.uint64(6))[:, None] | low).ravel()
    masks = np.bitwise_or.reduce(np.uint64(1) << low, axis=1)
    return keys[rng.permutation(len(keys))], np.unique(masks)


@pytest.fixture(scope="module")
def emu():
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    yield svd
    from dag_compression_fast_amd import _lib
    _lib._lib = None
    _lib._hip = None
    svd._default = None


def run_sizes(m, oracle, sizes, depth):
    rng = np.random.default_rng(0x1EAF)
    for count, bits in sizes:
        keys, masks = masked_leaves(rng, count, bits)
        print(f"[leaf-order] depth={depth} leaves={count} unique={len(masks)}", flush=True)
        dag = m.create_dag(keys, depth)
        got = dag.to_numpy()
        assert np.array_equal(got["leaves"], masks)
        assert_dag_equal(got, oracle.create_dag(keys, depth), f"{count} leaves")
        dag.free()


def test_leaf_order_on_the_cpu_emulator(emu, oracle):
    run_sizes(emu, oracle, [(1, 1), (2, 1), (63, 1), (700, 2), (1500, 4), (9000, 4)], 7)


@pytest.mark.gpu
def test_leaf_order_on_gpu(gpu, oracle):
    run_sizes(gpu, oracle, [(1, 1), (64, 2), (1024, 4), (1030, 4), (2100, 4), (66000, 5), (600000, 5)], 9)


@pytest.mark.gpu
def test_leaf_order_oversized_buckets(gpu):
    """Over 4M unique masks: buckets past one LDS sort are merged in global memory."""
    keys, masks = masked_leaves(np.random.default_rng(3), 9_000_000, 6)
    assert len(masks) > 8_000_000
    dag = gpu.create_dag(keys, 10)
    got = dag.to_numpy()
    assert np.array_equal(got["leaves"], masks)
    # The leaf level's children name their leaves: every parent's leaf masks, by
    # index, are its voxels' (checked through a flat-layout point query).
    words = gpu.create_final_dag(dag)
    probe = keys[:200_000]
    assert (gpu.query_voxels(words, 10, probe) == 1).all()
    dag.free()
