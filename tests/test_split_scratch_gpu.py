"""What a context's device memory grows by for a mixed batch split over its
walks' segments: nothing past the split's bound, where the batch takes its
segments in turn with the same bits, and nothing for walks from given normals,
which are not split."""
import ctypes

import numpy as np
import pytest

from conftest import DeviceArray

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert DeviceArray.hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_a_batch_past_the_bound_is_not_split(jne):
    dim, n, steps = 12, 700, 11_700  # 183 segments of 2,112 bytes each: 271 MB
    seeds = np.arange(1, n + 1, dtype=np.uint32)
    with jne.Engine(0) as eng:
        eng.eigenvalues_by_seed(4, dim, steps, seeds, precision=jne.PRECISIONS["mfma_bf16x2"])  # the other scratch
        before = free_bytes()
        full = eng.eigenvalues_by_seed(4, dim, steps, seeds, precision=jne.PRECISIONS["mfma_fp16x2"])
        assert before - free_bytes() < 1 << 24
        for at, m in ((0, 1), (300, 64), (n - 40, 40)):  # split
            got = eng.eigenvalues_by_seed(4, dim, steps, seeds[at:at + m], precision=jne.PRECISIONS["mfma_fp16x2"])
            assert np.array_equal(got, full[at:at + m]), (at, m)
        assert before - free_bytes() < 1 << 27


def test_given_normals_take_no_split_scratch(jne):
    dim, n, steps = 12, 600, 1500  # split by seed: 30 MB
    z = np.random.default_rng(3).standard_normal((n, steps, dim))
    with jne.Engine(0) as eng:
        eng.eigenvalues_from_normals(4, z, precision=jne.PRECISIONS["mfma_bf16x2"])  # the other scratch
        before = free_bytes()
        eng.eigenvalues_from_normals(4, z, precision=jne.PRECISIONS["mfma_fp16x2"])
        assert before - free_bytes() < 1 << 23
