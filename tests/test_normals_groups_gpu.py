"""The normals kernel at the edges of its launch shapes, bit for bit against the
CPU stream: walks of one wave, two waves and a whole group (64, 65, 128, 129 and
257 Philox calls), a last group that is not full, more rows of groups than one
launch covers, several calls per thread with a remainder, rows that are no
multiple of four floats, and outputs past the size from which they stream."""
import numpy as np
import pytest

from conftest import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,steps,n", [
    (1, 256, 5), (1, 260, 7), (4, 128, 3), (4, 129, 3), (4, 257, 2), (1, 255, 7), (3, 87, 5),
    (1, 4, 262_145), (1, 3, 262_145), (4, 771, 5003), (12, 1000, 5600), (3, 1003, 23_000),
])
def test_normals_launch_shapes(engine, O, dim, steps, n):
    seeds = np.arange(1, n + 1, dtype=np.uint32)
    seeds[-1] = 0xFFFFFFFF
    d_seeds, d_out = DeviceArray(seeds.nbytes), DeviceArray(n * steps * dim * 4)
    try:
        d_seeds.from_host(seeds)
        d_out.from_host(np.full(1024, np.nan, np.float32)[: n * steps * dim], max(0, n * steps * dim * 4 - 4096))
        engine.walk_normals_device(dim, steps, d_seeds.ptr, n, d_out.ptr)
        got = d_out.to_host((n, steps, dim), np.float32)
    finally:
        d_seeds.free()
        d_out.free()
    for k in sorted({0, 1, n // 2, n - 2, n - 1}):
        ref = O.walk_normals(int(seeds[k]), 0, dim, steps)
        assert np.array_equal(got[k].view(np.uint32), ref.view(np.uint32)), (dim, steps, k)
    assert np.isfinite(got).all()
