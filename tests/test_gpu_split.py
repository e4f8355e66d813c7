"""GPU parity of the split operands (three bf16 products a coordinate pair) on ordinary data,
which is what a base set without a half copy runs: UNG_HIP_NO_HALF=1, 32-bit and wide loads,
the register-query layout at 96 < d <= 128 and the restaged panels around it and in its place,
short, middle and long queues, long rows.  Rows bit for bit against the CPU oracle; few rows
may take the exact rescan, which would hide a wrong pre-selection."""
import os

import numpy as np
import pytest

import filtervectorcode_refactor_amd as F
from test_gpu_parity import _assert_rows_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["", "UNG_HIP_FORCE_WIDE", "UNG_HIP_NO_QREG"])
def split_ctx(request):
    names = ["UNG_HIP_NO_HALF"] + ([request.param] if request.param else [])
    old = {n: os.environ.get(n) for n in names}
    os.environ.update({n: "1" for n in names})
    try:
        c = F.HipContext(0)
    finally:
        for n, v in old.items():
            if v is None:
                del os.environ[n]
            else:
                os.environ[n] = v
    c.mode = request.param
    yield c
    c.close()


SIZES = [1, 130, 300, 2100, 700]  # three child groups, two target groups
GB = np.concatenate([[0, 0], np.cumsum(SIZES)]).astype(np.uint32)
OP, OI = np.array([0, 0, 2, 3, 5, 5, 5], np.uint32), np.array([4, 5, 4, 4, 5], np.uint32)


@pytest.mark.parametrize("d", [20, 33, 96, 97, 100, 128, 129, 384, 512])
@pytest.mark.parametrize("k", [1, 6, 12, 40])
def test_split_cross(split_ctx, oracle, d, k):
    print(f"split cross {split_ctx.mode} d={d} k={k}", flush=True)
    X = np.random.default_rng(11 * d + k).standard_normal((int(GB[-1]), d)).astype(np.float32)
    X[GB[4] + 7] = X[GB[4] + 3]
    split_ctx.prepare_vectors(X)
    ids, dist, size, st = split_ctx.cross_topk(GB, OP, OI, k)
    assert st["select_launches"] == 1 and st["fallback_rows"] <= 20
    ip, ii = F.in_neighbors(OP, OI)
    _assert_rows_equal(ids, dist, size, *oracle.cross_exact(X, GB, ip, ii, k), f"d={d} k={k}")


@pytest.mark.parametrize("d", [20, 100, 128, 200, 512])
@pytest.mark.parametrize("k", [6, 12, 32, 63])
def test_split_lists(split_ctx, oracle, d, k):
    print(f"split lists {split_ctx.mode} d={d} k={k}", flush=True)
    X = np.random.default_rng(13 * d + k).standard_normal((int(GB[-1]), d)).astype(np.float32)
    split_ctx.prepare_vectors(X)
    for g in (2, 4):
        ids, dist, st = split_ctx.group_knn([int(GB[g])], [SIZES[g - 1]], k)
        assert st["select_launches"] == 1 and st["fallback_rows"] <= 20
        _assert_rows_equal(ids, dist, None, *oracle.intra_exact(X, int(GB[g]), SIZES[g - 1], k), None, f"d={d} k={k}")
