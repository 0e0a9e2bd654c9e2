"""The mixed pass by seed draws a segment's normals as whole Philox calls and
lays its rows from them (dims whose segments are no whole number of 64-call
iterations) or stores each normal in its row (the others); from given normals
it always stores each in its row.  Both read the same normals in the same
order, so the results are equal bit for bit: at segments of one step, whole
segments and the partial last one, one to five segments (the calls drawn ahead
repeat after four), with walks enough to run each in a wave of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def outcome(jne, call):
    try:
        return call().tobytes()
    except jne.JneError as e:
        return e.code, str(e)


@pytest.mark.parametrize("prec", ["mfma_fp16x2", "mfma_bf16x2", "mfma_fp32"])
@pytest.mark.parametrize("dim", [5, 7, 8, 9, 10, 11, 12])
def test_by_seed_equals_from_normals(engine, jne, dim, prec):
    n = 801
    seeds = np.arange(1, n + 1, dtype=np.uint32)
    for steps in (dim + 2, 63, 64, 65, 129, 257, 321):
        z = engine.walk_normals(dim, steps, seeds).astype(np.float64)
        for model in (2, 3):
            # (of dim + 2 steps, 16 bits of the two-way bf16 split may leave no positive definite
            # matrix: then both forms say so, of the same walk)
            a = outcome(jne, lambda: engine.eigenvalues_by_seed(model, dim, steps, seeds, precision=jne.PRECISIONS[prec]))
            b = outcome(jne, lambda: engine.eigenvalues_from_normals(model, z, precision=jne.PRECISIONS[prec]))
            assert a == b, (dim, steps, model, prec)
            assert steps < 63 or isinstance(a, bytes), (dim, steps, model, prec)
