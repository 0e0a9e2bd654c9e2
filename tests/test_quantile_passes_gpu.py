"""Device percentiles at the edges of the passes: the largest array sorted in
LDS at once, one and many workgroups per pass, more values than the passes'
workgroups take in one stride; a NaN anywhere; the scratch reused by arrays of
other sizes in between."""
import numpy as np
import pytest

from test_quantile_gpu import PS, check, on_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4095, 4096, 4097, 16384, 16385, (1 << 20) + 1, (1 << 22) + 1, 9_000_001])
def test_pass_edges(engine, O, n):
    rng = np.random.default_rng(n)
    x = rng.chisquare(6, n)
    check(engine, O, x, [0.0, 0.5] + PS + [1.0])
    check(engine, O, x[: n // 3])
    check(engine, O, -x)


@pytest.mark.parametrize("n", [1000, 5000, 300_000])
def test_nan_anywhere(engine, jne, n):
    for at in (0, n // 2, n - 1):
        x = np.linspace(1.0, 2.0, n)
        x[at] = np.nan
        d = on_device(x)
        with pytest.raises(jne.JneError) as e:
            engine.percentiles_device(d.ptr, n, PS)
        assert e.value.code == jne.JNE_ERR_NUMERIC
        d.free()
