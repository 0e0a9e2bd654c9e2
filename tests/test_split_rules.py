"""The rules by which the moment passes choose a form, built for the host (CPU):
the split of a small mixed batch over its walks' segments, over every length the
entry points accept (2 to 2^30 steps), and the FP64 pass's forms."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "johansen-null-eigenspectra_amd", "csrc")

WAVES = [1, 2, 7, 100, 699, 700, 701, 5000]
STEPS = sorted({2, 63, 64, 256, 257, 1000, 10_000, 11_776, 12_000, 100_000, 1 << 30} |
               {x + d for x in (8_134_000, 16_776_960, 1 << 24, 1 << 25, 1 << 29) for d in (-64, -1, 0, 1, 64)})


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    so = str(tmp_path_factory.mktemp("split") / "libsplit.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC,
                    os.path.join(HERE, "split_rules.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.split_doubles.restype = ctypes.c_ulonglong
    return lib


def test_chunks_fit_the_grid(rule):
    """A split launch's chunks of segments are its grid's y dimension."""
    for steps in STEPS:
        for waves in WAVES:
            if rule.split_doubles(waves, steps):
                assert 1 < rule.chunks(steps) <= 65_535, (waves, steps)


def test_scratch_is_bounded(rule):
    """The segments' sums grow with the walk's length and stay with the context: 256 MiB at most."""
    for steps in STEPS:
        for waves in WAVES:
            assert 8 * rule.split_doubles(waves, steps) <= 1 << 28, (waves, steps)


def test_small_batches_are_split(rule):
    """The second kernel of a split costs the time of some segments: batches of walks of few
    segments are split only if they are small."""
    assert rule.split_doubles(1, 256) == 0 and rule.split_doubles(1, 257) == 5 * 264
    assert rule.split_doubles(100, 300) and not rule.split_doubles(400, 300)
    assert rule.split_doubles(300, 448) and not rule.split_doubles(600, 448)
    assert rule.split_doubles(650, 1000) and not rule.split_doubles(800, 1000)
    assert rule.split_doubles(701, 4000) and rule.split_doubles(800, 10_000) == 800 * 157 * 264
    assert rule.split_doubles(1000, 10_000) == 0


def test_unsplit_small_batches_of_dim_7_run_in_lane_groups(rule):
    """One lane per walk needs a wave per SIMD to be the better form at dim 7 (one walk of 1,000
    steps: 0.71 ms, in a group of seven lanes 0.21)."""
    for walks in (1, 9, 1000, 12_000, 50_000, 70_000, 90_000):
        assert rule.turn_lanes(7, walks) == 7, walks
    for walks in (60_000, 65_536, 131_072, 262_144):
        assert rule.turn_lanes(7, walks) == 1, walks
    assert [rule.turn_lanes(d, 100) for d in (1, 6, 8, 9, 10, 12)] == [1, 1, 2, 9, 5, 4]


@pytest.mark.parametrize("dim", range(1, 13))
def test_short_walks_are_not_split(rule, dim):
    """A split launch's second kernel and its sums cost the time of some steps: the shortest walks
    are never split, and those of one block in small batches only."""
    for walks in (1, 100, 3000, 12_000, 30_000, 65_000):
        for steps in range(2, 11):
            assert rule.turns(dim, steps, walks) == walks, (steps, walks)
    for steps in (2 * dim + 4, 40, 60):
        for walks in (30_000, 45_000, 100_000):
            if not (dim in (4, 6) and walks == 30_000):  # 1 to 3% either way
                assert rule.turns(dim, steps, walks) == walks, (steps, walks)


def test_forms_go_by_the_blocks_of_a_walk(rule):
    """A walk has at most 16 blocks: a few long walks are few waves."""
    assert [rule.form(d, 10_000, 100) for d in (1, 5, 8, 10)] == [0, 0, 0, 0]
    assert rule.form(5, 11_000_000, 1) == 0 and rule.form(8, 10_000, 1000) == 1
    assert rule.turns(8, 10_000, 1000) == 0 and rule.turns(12, 300, 20_000) == 0


def test_a_rest_is_split_where_that_is_faster(rule):
    """Dims 9-12 behind whole rounds of the GPU: a rest that the row form would take is left in turn
    where the two blocks of a walk just above 240 steps gain less than the split costs."""
    for dim, steps, walks in ((11, 241, 45_000), (11, 255, 75_000), (12, 241, 75_000), (10, 241, 45_000), (10, 300, 45_000)):
        assert rule.turns(dim, steps, walks) == walks, (dim, steps, walks)
    assert rule.turns(11, 1000, 100_000) == 98_304 and rule.turns(12, 1000, 100_000) == 98_304
    assert rule.turns(8, 241, 75_000) == 65_536 and rule.turns(5, 241, 140_000) == 131_072


def test_dim_7_is_split_where_that_beats_its_lane_groups(rule):
    for steps, walks in ((400, 36_000), (480, 36_000), (480, 45_000), (480, 70_000)):
        assert rule.turns(7, steps, walks) == walks, (steps, walks)
    for steps, walks in ((480, 50_000), (480, 30_000), (1000, 36_000), (1000, 55_000), (333, 50_001)):
        assert rule.turns(7, steps, walks) == 0, (steps, walks)
