"""svdag_dag_to_host reports what it could not copy: a refused kernel launch or
copy is an error, and the result holds nothing then.  On the CPU emulator,
which refuses a chosen launch or copy."""
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
