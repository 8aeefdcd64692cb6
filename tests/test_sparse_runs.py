"""Batched builds of few keys in many chunks, most chunks empty: the leaf
reduce's runs are one per chunk with keys (chunk depth 7 has 8 cells a chunk),
more of them than the key sort has tile counts.  Chunk counts around the 512
and 640 words that one tile's counts and what lies behind them hold, up to the
most that the cells take (1024); keys around one tile (4096).  Integer output,
equal to the oracle's bit for bit; the emulator runs both block orders."""
import numpy as np
import pytest

from dagcheck import assert_dag_equal

DEPTH, LEVELS = 7, 4
SLOTS = 8 ** LEVELS
# (chunks with keys, keys in all)
SHAPES = ((512, 1024), (513, 1026), (640, 4096), (641, 4096), (1000, 2000), (1000, 4000), (1000, 4097), (1024, 4096),
          (1025, 4100))


def chunks_of(rng, live, n):
    ids = np.sort(rng.choice(SLOTS, size=live, replace=False))
    sizes = np.full(live, n // live)
    sizes[:n % live] += 1
    return {int(i): rng.integers(0, 1 << (3 * DEPTH), size=int(k), dtype=np.uint64) for i, k in zip(ids, sizes)}


def union_of(chunks):
    return np.concatenate([(np.uint64(i) << np.uint64(3 * DEPTH)) | c for i, c in sorted(chunks.items())])


def run_shapes(m, oracle, shapes):
    rng = np.random.default_rng(0x5A125)
    for live, n in shapes:
        chunks = chunks_of(rng, live, n)
        offsets = np.zeros(SLOTS + 1, dtype=np.uint64)
        offsets[1:] = np.cumsum([len(chunks.get(i, ())) for i in range(SLOTS)])
        keys = np.concatenate([c for _, c in sorted(chunks.items())])
        print(f"[sparse] {live} of {SLOTS} chunks, {n} keys", flush=True)
        dag = m.create_dag_batched(keys, offsets, DEPTH)
        assert_dag_equal(dag.to_numpy(), oracle.create_dag(union_of(chunks), DEPTH + LEVELS), f"{live} chunks, {n} keys")
        dag.free()


def run_served(m, oracle):
    from dag_compression_fast_amd import serve
    chunks = chunks_of(np.random.default_rng(0x5A126), 1000, 4000)
    server = serve.ChunkServer(DEPTH, LEVELS, max_nodes=1 << 16)
    try:
        print("[sparse] a served round of 1000 chunks", flush=True)
        results = server.run([serve.Request(j, i, c, 0.0) for j, (i, c) in enumerate(chunks.items())])
        assert max(r.round for r in results) == 0
        assert_dag_equal(server.dag().to_numpy(), oracle.create_dag(union_of(chunks), DEPTH + LEVELS), "served")
    finally:
        server.close()


@pytest.fixture(scope="module")
def emu():
    import ctypes
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    yield svd, ctypes.CDLL(emu_ctypes.EMU_LIB)
    from dag_compression_fast_amd import _lib
    svd._default = None  # the emulator's context goes before its library
    _lib._lib = None
    _lib._hip = None


def test_sparse_runs_on_the_cpu_emulator(emu, oracle):
    run_shapes(emu[0], oracle, ((513, 1026), (641, 4096), (1000, 2000), (1000, 4097), (1024, 4096)))
    run_served(emu[0], oracle)


def test_sparse_runs_in_reverse_block_order(emu, oracle):
    emu[1].emu_set_schedule(1)
    try:
        run_shapes(emu[0], oracle, ((1000, 2000),))
    finally:
        emu[1].emu_set_schedule(0)


@pytest.mark.gpu
def test_sparse_runs_on_gpu(gpu, oracle):
    run_shapes(gpu, oracle, SHAPES)
    run_served(gpu, oracle)
