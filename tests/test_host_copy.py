"""svdag_dag_to_host reports what it could not copy: a refused kernel launch or
copy is an error, and the result holds nothing then.  Its kernel reads memory of
the context's own device only, and an array that the DAG does not have stays
null.  DAGs of 160 MiB or more are copied array by array.  On the CPU emulator,
which refuses a chosen launch or copy and counts launches."""
import ctypes

import numpy as np
import pytest


@pytest.fixture(scope="module")
def emu():
    import emu_ctypes
    svd = emu_ctypes.use_emulator()
    lib = ctypes.CDLL(emu_ctypes.EMU_LIB)
    lib.emu_launch_count.restype = ctypes.c_uint64
    yield svd, lib
    from dag_compression_fast_amd import _lib
    svd._default = None
    _lib._lib = None
    _lib._hip = None


def a_dag(svd, depth=6):
    return svd.create_dag(np.random.default_rng(4).integers(0, 1 << (3 * depth), size=3000, dtype=np.uint64), depth)


def to_host(svd, raw):
    """(return code, host DAG) of svdag_dag_to_host."""
    from dag_compression_fast_amd import _lib
    out = _lib.SvdagDag()
    return _lib.lib().svdag_dag_to_host(svd.default_context().handle, ctypes.byref(raw), ctypes.byref(out)), out


def assert_refused(svd, rc, out):
    from dag_compression_fast_amd import _lib
    assert rc != 0
    assert b"copy to host failed" in _lib.lib().svdag_last_error()
    assert not out.storage and not out.leaves and out.num_leaves == 0
    assert all(not out.levels[l].hashes and out.levels[l].num_nodes == 0 for l in range(out.num_levels))


def off_boundary(dag):
    """The DAG with its leaves 8 bytes off a 16-byte boundary (a copy of its
    own beside the kernel's), and what keeps them."""
    from dag_compression_fast_amd import _lib
    raw = _lib.SvdagDag.from_buffer_copy(dag.raw)
    n = int(raw.num_leaves)
    room = np.zeros(n + 3, dtype=np.uint64)
    at = room.ctypes.data + (16 - room.ctypes.data % 16) + 8
    ctypes.memmove(at, raw.leaves, 8 * n)
    raw.leaves = at
    return raw, room


def test_a_refused_launch_is_an_error(emu):
    svd, lib = emu
    dag = a_dag(svd)
    lib.emu_fail_launch(1)
    try:
        assert_refused(svd, *to_host(svd, dag.raw))
    finally:
        lib.emu_fail_launch(0)
    rc, out = to_host(svd, dag.raw)  # and the next call is not blamed
    assert rc == 0
    svd.Dag(out, dag.ctx).free()


def test_a_refused_copy_is_an_error(emu):
    svd, lib = emu
    dag = a_dag(svd)
    raw, keep = off_boundary(dag)
    lib.emu_fail_copy(1)
    try:
        assert_refused(svd, *to_host(svd, raw))
    finally:
        lib.emu_fail_copy(0)
    rc, out = to_host(svd, raw)
    assert rc == 0
    got = svd.Dag(out, dag.ctx)
    assert np.array_equal(got.to_numpy()["leaves"], dag.to_numpy()["leaves"])
    got.free()


def test_memory_of_another_device_is_not_read_by_the_kernel(emu):
    svd, lib = emu
    other = svd.Context()
    try:
        dag = svd.create_dag(np.arange(0, 200000, 37, dtype=np.uint64), 6, ctx=other)  # not in the default context's pool
        for device, kernels in ((0, 1), (1, 0)):
            lib.emu_set_pointer_device(device)
            before = lib.emu_launch_count()
            rc, out = to_host(svd, dag.raw)
            assert rc == 0 and lib.emu_launch_count() - before == kernels
            got, want = svd.Dag(out, svd.default_context()), dag.to_numpy()
            for a, b in zip(got.to_numpy()["levels"], want["levels"]):
                assert all(np.array_equal(a[k], b[k]) for k in b)
            got.free()
        dag.free()
    finally:
        lib.emu_set_pointer_device(0)
        other.close()


def test_an_array_that_is_not_there_stays_null(emu):
    svd, _ = emu
    from dag_compression_fast_amd import _lib
    dag = a_dag(svd)
    raw = _lib.SvdagDag.from_buffer_copy(dag.raw)
    for l in range(raw.num_levels):
        raw.levels[l].hashes = None
    rc, out = to_host(svd, raw)
    assert rc == 0
    assert all(not out.levels[l].hashes for l in range(out.num_levels))
    for l in range(out.num_levels):
        out.levels[l].hashes = out.levels[l].children  # to_numpy reads every array
    got, want = svd.Dag(out, dag.ctx), dag.to_numpy()
    assert np.array_equal(got.to_numpy()["leaves"], want["leaves"])
    for a, b in zip(got.to_numpy()["levels"], want["levels"]):
        assert np.array_equal(a["masks"], b["masks"]) and np.array_equal(a["children"], b["children"])
    got.free()


@pytest.mark.parametrize("words, kernels", [((160 << 17) - 9, 1), ((160 << 17) - 8, 0)])
def test_large_dags_leave_by_the_copy_engine(emu, words, kernels):
    # Leaves alone, and the 16 + 48 bytes of padding a one-level DAG is given.
    svd, lib = emu
    from dag_compression_fast_amd import _lib
    leaves = svd.DeviceBuffer.from_numpy(np.arange(words, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15))
    raw = _lib.SvdagDag()
    raw.num_levels, raw.location, raw.num_leaves, raw.leaves = 1, svd.SVDAG_DEVICE, words, leaves.address
    before = lib.emu_launch_count()
    rc, out = to_host(svd, raw)
    assert rc == 0 and lib.emu_launch_count() - before == kernels
    got = svd.Dag(out, svd.default_context())
    assert np.array_equal(got.to_numpy()["leaves"], leaves.to_numpy(np.uint64, words))
    got.free()
    leaves.free()
