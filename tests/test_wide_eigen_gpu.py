"""The eigen solve of dims 13..32: every dim and model against the oracle at the
parity bar (33 rows at dim 32 in models 1 and 3, where the rows of S10 and of M
take one lane more than a wave has), walks in any place of a batch give the same
bits, and a walk whose S11 is not positive definite is NaN in every entry."""
import numpy as np
import pytest

from conftest import DeviceArray, assert_eigs_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", range(13, 33))
def test_every_dim_and_model(engine, O, dim):
    seeds = np.array([1, 7, 0xFFFFFFFF], dtype=np.uint32)
    for model in range(5):
        for steps in (3 * dim, 401):
            got = engine.eigenvalues_by_seed(model, dim, steps, seeds)
            assert_eigs_close(got, O.walks_by_seed_c(model, dim, steps, seeds), 1e-9, f"{model} {dim} {steps}")


@pytest.mark.parametrize("dim,n", [(13, 1), (16, 7), (24, 1001), (32, 2051)])
def test_same_bits_in_any_place(engine, dim, n):
    seeds = np.arange(1, n + 1, dtype=np.uint32)
    for model in (0, 3):
        full = engine.eigenvalues_by_seed(model, dim, 150, seeds)
        for at, m in ((0, 1), (n // 2, 1), (n - 1, 1), (n // 3, n // 3 + 1)):
            assert np.array_equal(full[at:at + m], engine.eigenvalues_by_seed(model, dim, 150, seeds[at:at + m]))


@pytest.mark.parametrize("dim,model", [(13, 0), (20, 1), (24, 4), (32, 3)])
def test_not_positive_definite_is_nan(engine, jne, dim, model):
    n, nf = 9, jne.num_eigenvalues(model, dim)
    d_seeds, d_out = DeviceArray(4 * n), DeviceArray(8 * n * nf)
    try:
        d_seeds.from_host(np.arange(1, n + 1, dtype=np.uint32))
        d_out.from_host(np.zeros((n, nf)))
        engine.eigenvalues_by_seed_device(model, dim, 4, d_seeds.ptr, n, d_out.ptr)
        got = d_out.to_host((n, nf), np.float64)
    finally:
        d_seeds.free()
        d_out.free()
    bad = np.isnan(got)
    assert (bad.all(axis=1) == bad.any(axis=1)).all() and bad.any()
