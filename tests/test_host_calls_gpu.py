"""Host calls on both sides of the size (1 MiB of seeds and eigenvalues) up to
which the kernels read and write pinned host memory: the same bits as the device
entry point, and the NaN check of a small call."""
import numpy as np
import pytest

from conftest import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,dim,n", [(2, 5, 1), (2, 5, 23831), (2, 5, 23832), (1, 1, 3), (3, 32, 700),
                                         (4, 12, 10485), (4, 12, 10486)])
def test_host_equals_device(engine, jne, model, dim, n):
    steps = 60
    nf = jne.num_eigenvalues(model, dim)
    seeds = np.arange(3, 3 + n, dtype=np.uint32)
    d_seeds, d_out = DeviceArray(seeds.nbytes), DeviceArray(n * nf * 8)
    try:
        d_seeds.from_host(seeds)
        engine.eigenvalues_by_seed_device(model, dim, steps, d_seeds.ptr, n, d_out.ptr)
        want = d_out.to_host((n, nf), np.float64)
    finally:
        d_seeds.free()
        d_out.free()
    first = engine.eigenvalues_by_seed(model, dim, steps, seeds)
    again = engine.eigenvalues_by_seed(model, dim, steps, seeds[::-1].copy())
    assert np.array_equal(first, want) and np.array_equal(again[::-1], want)


def test_small_call_names_the_nan_walk(engine, jne):
    # 3 steps of 12 components: S11 has rank 3, no walk's is positive definite
    with pytest.raises(jne.JneError) as e:
        engine.eigenvalues_by_seed(0, 12, 3, np.arange(1, 6, dtype=np.uint32))
    assert e.value.code == jne.JNE_ERR_NUMERIC and "walk 0" in str(e.value)
