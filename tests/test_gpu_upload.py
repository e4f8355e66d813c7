"""GPU tests of the upload: the norms, the maxima and both operand sets of rows at the ends of
its passes (four and two rows a wave, grid-stride past 32,768 and 16,384 rows), the largest
coordinate in the last row; lists of the last rows bit for bit against the CPU oracle, on
both operand sets.  The resident set takes two allocations (five made a small upload half as
long again)."""
import os

import numpy as np
import pytest

import filtervectorcode_refactor_amd as F
from test_gpu_parity import _assert_rows_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["", "UNG_HIP_NO_HALF"])
def ctx(request):
    if request.param:
        os.environ[request.param] = "1"
    try:
        c = F.HipContext(0)
    finally:
        if request.param:
            del os.environ[request.param]
    c.most = 1 if request.param else 2
    yield c
    c.close()


@pytest.mark.parametrize("n", [2, 3, 5, 9, 131, 16383, 16385, 32767, 32769, 32771])
@pytest.mark.parametrize("d", [1, 65, 130])
def test_row_ends(ctx, oracle, n, d):
    print(f"upload n={n} d={d}", flush=True)
    X = np.random.default_rng(n + d).standard_normal((n, d)).astype(np.float32)
    X[-1, -1] = 1.3 * np.abs(X).max()
    ctx.prepare_vectors(X)  # (its first call may also allocate the download's pinned memory)
    assert ctx.prepare_vectors(X)["allocations"] == ctx.most
    m = min(n, 300)
    for k in (8, 32):
        ids, dist, st = ctx.group_knn([n - m], [m], k)
        _assert_rows_equal(ids, dist, None, *oracle.intra_exact(X, n - m, m, k), None, f"n={n} d={d} k={k}")
        assert st["fallback_rows"] <= 20 or d == 1
