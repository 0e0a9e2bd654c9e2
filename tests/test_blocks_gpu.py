"""The FP64 moment pass's forms: a walk's blocks of steps taken in turn by one
lane group (whole rounds of a batch that fills the GPU), or each block with a lane
group, a lane per component, or a wave of its own.  The blocks' sums and the order they are added
in are the same in every form, so a batch, its pieces and single walks give
the same bits; each length is also held to the C oracle at 1e-9."""
import numpy as np
import pytest

from conftest import assert_eigs_close

pytestmark = pytest.mark.gpu

# one walk per lane up to dim 7 (64 per wave at 4, 4, 4, 3, 2, 2, 2 waves per SIMD), lane groups above
ROUND = {1: 262144, 2: 262144, 3: 262144, 4: 196608, 5: 131072, 6: 131072, 7: 131072, 8: 65536, 9: 28672, 10: 36864,
         11: 32768, 12: 32768}


@pytest.mark.parametrize("dim,steps", [(1, 2)] + [(d, t) for d in range(1, 13) for t in (239, 241, 483)])
def test_forms_give_the_same_bits(engine, O, dim, steps):
    model = 0 if steps == 2 else dim % 5
    n = ROUND[dim] + 50001  # a whole round (blocks in turn) and a split rest
    seeds = np.arange(11, 11 + n, dtype=np.uint32)
    full = engine.eigenvalues_by_seed(model, dim, steps, seeds)
    for at, m in [(0, 50000), (n - 9000, 9000), (9, 3000), (5, 100), (n - 1, 1)]:
        part = engine.eigenvalues_by_seed(model, dim, steps, seeds[at:at + m])
        assert np.array_equal(part, full[at:at + m]), (dim, steps, at, m)
    ends = np.r_[0:3, n - 3:n]
    assert_eigs_close(full[ends], O.walks_by_seed_c(model, dim, steps, seeds[ends]), 1e-9, f"dim {dim} steps {steps}")


@pytest.mark.parametrize("dim", [1, 4, 7, 8, 12])
def test_long_blocks(engine, O, dim):
    """T > 3,840: blocks of more than 240 steps, the last one partial; from-normals and by-seed."""
    steps, seeds = 7999, np.arange(1, 2501, dtype=np.uint32)
    full = engine.eigenvalues_by_seed(4, dim, steps, seeds)
    assert np.array_equal(full[7:9], engine.eigenvalues_by_seed(4, dim, steps, seeds[7:9]))
    assert_eigs_close(full[:2], O.walks_by_seed_c(4, dim, steps, seeds[:2]), 1e-9, f"dim {dim}")
    z = engine.walk_normals(dim, steps, seeds[:40]).astype(np.float64)
    assert np.array_equal(engine.eigenvalues_from_normals(4, z), full[:40])


@pytest.mark.parametrize("dim", [13, 16, 17, 20, 21, 24, 25, 28, 29, 32])
@pytest.mark.parametrize("steps", [241, 503, 4999])
def test_wide_forms_give_the_same_bits(engine, O, dim, steps):
    """Dims 13..32: one wave per walk taking its blocks in turn, or one per block of a walk; every
    padded class at both ends."""
    n = (4100 if dim <= 24 else 3100) + 300
    seeds = np.arange(5, 5 + n, dtype=np.uint32)
    full = engine.eigenvalues_by_seed(dim % 5, dim, steps, seeds)
    for at, m in [(0, 700), (n - 3, 3), (17, 1)]:
        assert np.array_equal(engine.eigenvalues_by_seed(dim % 5, dim, steps, seeds[at:at + m]), full[at:at + m])
    ends = np.r_[0:2, n - 2:n]
    assert_eigs_close(full[ends], O.walks_by_seed_c(dim % 5, dim, steps, seeds[ends]), 1e-9, f"dim {dim} steps {steps}")


@pytest.mark.parametrize("dim", range(1, 13))
@pytest.mark.parametrize("steps", [257, 512, 1003])
def test_mixed_split_gives_the_same_bits(engine, jne, dim, steps):
    """The fp16x2 pass split over its walks' segments (batches of few waves) and taking them in turn;
    from-normals always takes them in turn."""
    p = jne.PRECISIONS["mfma_fp16x2"]
    n = 1300 * (12 // dim if 12 % dim == 0 else 1)  # packed dims: 12 / dim walks per wave
    seeds = np.arange(1, 1 + n, dtype=np.uint32)
    full = engine.eigenvalues_by_seed(dim % 5, dim, steps, seeds, precision=p)
    for at, m in [(0, n // 2), (3, 1), (n - 7, 7)]:
        got = engine.eigenvalues_by_seed(dim % 5, dim, steps, seeds[at:at + m], precision=p)
        assert np.array_equal(got, full[at:at + m]), (dim, steps, at, m)
    z = engine.walk_normals(dim, steps, seeds[:9]).astype(np.float64)
    assert np.array_equal(engine.eigenvalues_from_normals(dim % 5, z, precision=p), full[:9])


@pytest.mark.parametrize("dim,n", [(1, 70_000), (2, 90_000), (6, 66_000), (7, 52_500), (9, 20_000), (10, 40_000), (12, 20_000)])
@pytest.mark.parametrize("steps", [264, 265, 333])
def test_rounds_and_rests_give_the_same_bits(engine, O, dim, n, steps):
    """Second blocks of 24, 25 and 93 steps; whole rounds, rests taken in turn with them and rests
    split, against the small batches' forms and the oracle."""
    seeds = np.arange(9, 9 + n, dtype=np.uint32)
    full = engine.eigenvalues_by_seed(2, dim, steps, seeds)
    for at, m in [(0, 1), (n // 2, 700), (n - 2, 2)]:
        assert np.array_equal(full[at:at + m], engine.eigenvalues_by_seed(2, dim, steps, seeds[at:at + m])), (at, m)
    assert_eigs_close(full[:2], O.walks_by_seed_c(2, dim, steps, seeds[:2]), 1e-9, f"dim {dim}")
