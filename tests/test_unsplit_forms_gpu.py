"""FP64 calls that are not split: captured ones, and allocation-free ones whose
walks leave too little of the fixed scratch for the blocks' sums.  At dim 7 small
ones take their blocks in turn in groups of seven lanes, larger ones in a lane
per walk; every form gives the eager call's bits."""
import ctypes

import numpy as np
import pytest

from conftest import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,steps,n", [(7, 100, 5000), (7, 239, 55_000), (7, 241, 1), (7, 241, 10), (7, 500, 55_001),
                                         (7, 483, 65_537), (7, 4000, 9), (7, 300, 95_001), (1, 500, 700), (6, 500, 700),
                                         (8, 500, 700), (9, 500, 700), (12, 500, 700)])
def test_captured_call_gives_the_eager_bits(jne, dim, steps, n):
    hip = DeviceArray.hip()
    d_seeds, d_out = DeviceArray(4 * n), DeviceArray(8 * n * dim)
    st = DeviceArray.stream()
    graph, ex, stream = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p(st)
    try:
        with jne.Engine(0) as engine:
            d_seeds.from_host(np.arange(1, n + 1, dtype=np.uint32))

            def call():
                engine.eigenvalues_by_seed_device(4, dim, steps, d_seeds.ptr, n, d_out.ptr, hip_stream=st)

            call()
            want = d_out.to_host((n, dim), np.float64)
            assert np.isfinite(want).all()
            assert hip.hipStreamBeginCapture(stream, 2) == 0  # relaxed
            call()
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
            assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
            for _ in range(3):
                d_out.from_host(np.zeros((n, dim)))
                assert hip.hipGraphLaunch(ex, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
                assert np.array_equal(d_out.to_host((n, dim), np.float64), want)
    finally:
        if ex:
            hip.hipGraphExecDestroy(ex)
        if graph:
            hip.hipGraphDestroy(graph)
        d_seeds.free()
        d_out.free()
        DeviceArray.destroy_stream(st)


@pytest.mark.parametrize("steps", [300, 1000])
def test_allocation_free_call_gives_the_same_bits(jne, engine, steps):
    n = 40_000  # leaves 13 MB of the scratch: the blocks' sums would take 67 MB and more
    d_seeds, d_a, d_b = DeviceArray(4 * n), DeviceArray(56 * n), DeviceArray(56 * n)
    try:
        d_seeds.from_host(np.arange(1, n + 1, dtype=np.uint32))
        engine.eigenvalues_by_seed_device(4, 7, steps, d_seeds.ptr, n, d_a.ptr)
        engine.eigenvalues_by_seed_device_noalloc(4, 7, steps, d_seeds.ptr, n, d_b.ptr)
        engine.synchronize()
        assert np.array_equal(d_a.to_host((n, 7), np.float64), d_b.to_host((n, 7), np.float64))
    finally:
        for a in (d_seeds, d_a, d_b):
            a.free()
