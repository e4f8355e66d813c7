"""GPU parity of the half-precision pre-selection (one fp16 product per coordinate pair,
rows certified against the base set's measured rounding error) where it can go wrong: row
widths around its 64-dimension chunks, base sets that its error bound cannot certify (the
call is repeated on the split operands), coordinates outside its range, and sets it holds
exactly.  Every row bit for bit against the CPU oracle."""
import numpy as np
import pytest

import filtervectorcode_refactor_amd as F
from test_gpu_parity import _assert_rows_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = F.HipContext(0)
    yield c
    c.close()


def _vectors(kind, rng, n, d):
    X = rng.standard_normal((n, d)).astype(np.float32)
    if kind == "bytes":
        return rng.integers(0, 256, size=(n, d)).astype(np.float32)
    if kind == "far":  # one cluster of radius ~0.3 sqrt(d) at norm 50
        c = rng.standard_normal(d)
        return (X * 0.3 + 50.0 * c / np.linalg.norm(c)).astype(np.float32)
    if kind == "mixed":  # a few rows a billion times larger than the rest
        X *= np.float32(1e-3)
        X[:: n // 7] *= np.float32(1e9)
        return X
    return X * np.float32({"normal": 1.0, "huge": 1e13, "tiny": 1e-13}[kind])


@pytest.mark.parametrize("kind,d", [("normal", 1), ("normal", 33), ("normal", 64), ("normal", 65), ("normal", 127),
                                    ("normal", 129), ("normal", 200), ("bytes", 64), ("bytes", 128), ("far", 128),
                                    ("far", 96), ("mixed", 40), ("huge", 128), ("tiny", 128)])
@pytest.mark.parametrize("k", [6, 12])
def test_half_preselect(ctx, oracle, kind, d, k):
    print(f"half pre-selection {kind} d={d} k={k}", flush=True)
    rng = np.random.default_rng(7 * d + k)
    sizes = [1, 130, 300, 2100, 700]  # three child groups, two target groups
    gb = np.zeros(len(sizes) + 2, np.uint32)
    gb[2:] = np.cumsum(sizes)
    op = np.array([0, 0, 2, 3, 5, 5, 5], np.uint32)
    oi = np.array([4, 5, 4, 4, 5], np.uint32)
    X = _vectors(kind, rng, int(gb[-1]), d)
    ctx.prepare_vectors(X)
    ids, dist, size, st = ctx.cross_topk(gb, op, oi, k)
    ip, ii = F.in_neighbors(op, oi)
    _assert_rows_equal(ids, dist, size, *oracle.cross_exact(X, gb, ip, ii, k), f"{kind} d={d} k={k}")
    if kind == "far":  # half: 2 rho (|q| + R) ~ 2.5, above most rows' D16 - D6 ~ 1; split: ~0.2
        assert st["select_launches"] == 2 and st["fallback_rows"] < 200
    elif kind in ("normal", "bytes", "huge", "tiny") and d > 1:
        assert st["select_launches"] == 1
    ids, dist, st = ctx.group_knn([int(gb[4])], [sizes[3]], 32)
    _assert_rows_equal(ids, dist, None, *oracle.intra_exact(X, int(gb[4]), sizes[3], 32), None, f"{kind} lists d={d}")
