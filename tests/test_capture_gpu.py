"""A captured call of the device entry point allocates nothing: after a larger
batch that needed no room for block sums, a smaller one that would be split is
captured, replayed between eager calls, and gives the eager results' bits."""
import ctypes

import numpy as np
import pytest

from conftest import DeviceArray

pytestmark = pytest.mark.gpu


def test_capture_after_a_larger_batch(jne):
    dim, steps, warm, n = 6, 600, 131_072, 66_000
    hip = DeviceArray.hip()
    engine = jne.Engine(0)
    seeds = np.arange(1, warm + 1, dtype=np.uint32)
    d_seeds, d_out = DeviceArray(seeds.nbytes), DeviceArray(warm * dim * 8)
    st = DeviceArray.stream()
    graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
    stream = ctypes.c_void_p(st)
    try:
        d_seeds.from_host(seeds)

        def call(m):
            engine.eigenvalues_by_seed_device(0, dim, steps, d_seeds.ptr, m, d_out.ptr, hip_stream=st)

        call(warm)
        want = d_out.to_host((warm, dim), np.float64)[:n]
        assert hip.hipStreamBeginCapture(stream, 2) == 0  # relaxed
        call(n)
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
        for _ in range(3):
            d_out.from_host(np.zeros((n, dim)))
            assert hip.hipGraphLaunch(ex, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
            assert np.array_equal(d_out.to_host((n, dim), np.float64), want)
            call(777)
            assert hip.hipStreamSynchronize(stream) == 0
            assert np.array_equal(d_out.to_host((777, dim), np.float64), want[:777])
    finally:
        if ex:
            hip.hipGraphExecDestroy(ex)
        if graph:
            hip.hipGraphDestroy(graph)
        d_seeds.free()
        d_out.free()
        DeviceArray.destroy_stream(st)
