"""The voxelizer's units of work (at most 8 columns of one row): triangles whose
rows hold from one to a few units, with full and partial last units, and tiles
of units (256) that end inside a triangle.  The voxels equal the host rule's,
and the keys come out in the same order on every call."""
import numpy as np
import pytest


def run_legs(m, legs, depth):
    for leg in legs:
        for axis in range(3):
            # Two right triangles that fill a leg x leg square across `axis`.
            a, b, c, d = (3.25, 2.5), (3.25 + leg, 2.5), (3.25, 2.5 + leg), (3.25 + leg, 2.5 + leg)
            tris = np.zeros((2, 3, 3))
            for t, corners in enumerate(((a, b, c), (d, c, b))):
                for k, (p, q) in enumerate(corners):
                    tris[t, k, axis], tris[t, k, (axis + 1) % 3], tris[t, k, (axis + 2) % 3] = 5.3 + 0.1 * k, p, q
            want = m.gen_voxelize(tris, depth)
            got = []
            for _ in range(2):
                buf, n = m.voxelize_triangles(tris, depth)
                got.append(buf.to_numpy(np.uint64, n))
                buf.free()
            assert np.array_equal(got[0], got[1])
            assert np.array_equal(np.unique(got[0]), want), (leg, axis)


def test_units_on_the_cpu_emulator():
    import emu_ctypes
    m = emu_ctypes.use_emulator()
    try:
        run_legs(m, (0.6, 5.0, 6.0, 7.0, 13.0, 14.0, 15.5, 40.0), 6)
    finally:
        from dag_compression_fast_amd import _lib
        import dag_compression_fast_amd as svd
        _lib._lib = None
        _lib._hip = None
        svd._default = None


@pytest.mark.gpu
def test_units_on_gpu(gpu):
    run_legs(gpu, (0.6, 5.0, 6.0, 7.0, 13.0, 14.0, 15.5, 40.0, 500.0), 10)
