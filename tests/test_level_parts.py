"""Level builds and extracts over parts of tiles (a count per part, summed by
the workgroups), and the merge whose top levels take one workgroup (up to 8^4
chunks) or the hashed levels (8^5).  Leaf counts sit at the edges of a tile
(512 children), of the leaf order in one workgroup (4096 keys) and of the
estimated table (32768), with one and with eight leaves a parent; inputs that leave all
but one part empty and levels of one node are among them."""
import numpy as np
import pytest

from dagcheck import assert_dag_equal


def check(m, oracle, keys, depth):
    print(f"[parts] depth {depth} {len(keys)} keys", flush=True)
    dag = m.create_dag(keys, depth)
    exp = oracle.create_dag(keys, depth)
    assert_dag_equal(dag.to_numpy(), exp, f"depth {depth} {len(keys)} keys")
    assert dag.pre_dedup == exp["pre_dedup"]
    assert np.array_equal(m.create_final_dag(dag), oracle.create_final_dag(exp))
    dag.free()


def run_builds(m, oracle):
    rng = np.random.default_rng(0x9A77)
    for leaves in (1, 8, 511, 512, 513, 1023, 1024, 1025, 2047, 2049, 4095, 4096, 4097, 16385, 32769):
        # Consecutive leaves (8 a parent), and one leaf a parent.
        for step, depth in ((1, 8), (8, 9), (64, 9)):
            codes = np.arange(leaves, dtype=np.uint64) * np.uint64(step) + np.uint64(step - 1)
            codes = codes[codes < (1 << (3 * depth - 6))]
            keys = (codes << np.uint64(6)) | rng.integers(0, 64, size=len(codes), dtype=np.uint64)
            check(m, oracle, keys[rng.permutation(len(keys))], depth)


def run_merges(m, oracle):
    rng = np.random.default_rng(0x9A78)
    for k in range(6):
        num = 8 ** k
        live = np.unique(np.concatenate(([0, num - 1], rng.integers(0, num, size=5))))
        chunks = {int(i): rng.integers(0, 1 << 18, size=200, dtype=np.uint64) for i in live}
        empty = np.empty(0, dtype=np.uint64)
        print(f"[parts] merge of {len(live)} in {num} chunks", flush=True)
        dags = [m.create_dag(chunks.get(i, empty), 6) for i in range(num)]
        merged = m.merge_dags(dags)
        union = np.concatenate([(np.uint64(i) << np.uint64(18)) | c for i, c in chunks.items()])
        assert_dag_equal(merged.to_numpy(), oracle.create_dag(union, 6 + k), f"merge of 8^{k}")


@pytest.fixture(scope="module")
def emu():
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    yield svd
    from dag_compression_fast_amd import _lib
    _lib._lib = None
    _lib._hip = None
    svd._default = None


def test_parts_on_the_cpu_emulator(emu, oracle):
    run_builds(emu, oracle)
    run_merges(emu, oracle)


@pytest.mark.gpu
def test_parts_on_gpu(gpu, oracle):
    run_builds(gpu, oracle)
    run_merges(gpu, oracle)
