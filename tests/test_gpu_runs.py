"""GPU parity of the item order of long operand rows (d > 448): runs of 64 consecutive items
per XCD with take-over at the end of the list, and cross unions cut into up to 4 splits of at
least 2048 candidates.  Either side of the row width and of each split count, item counts
below, at and past a round of 8 runs, short and long queues.  Rows bit for bit against the
CPU oracle."""
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


def _check(ctx, oracle, sizes, edges, d, k, name):
    """sizes[g - 1] points in group g, edges {child: targets}."""
    print(f"runs {name} d={d} k={k}", flush=True)
    G = len(sizes)
    gb = np.zeros(G + 2, np.uint32)
    gb[2:] = np.cumsum(sizes)
    op, oi = np.zeros(G + 2, np.uint32), []
    for g in range(1, G + 1):
        oi += edges.get(g, [])
        op[g + 1] = len(oi)
    oi = np.array(oi, np.uint32)
    X = np.random.default_rng(d + k).standard_normal((int(gb[-1]), d)).astype(np.float32)
    ctx.prepare_vectors(X)
    ids, dist, size, _ = ctx.cross_topk(gb, op, oi, k)
    ip, ii = F.in_neighbors(op, oi)
    _assert_rows_equal(ids, dist, size, *oracle.cross_exact(X, gb, ip, ii, k), name)
    return X, gb


@pytest.mark.parametrize("k", [6, 12, 40])
@pytest.mark.parametrize("d", [448, 449, 512, 770])
def test_split_edges(ctx, oracle, d, k):
    # unions of 1, 1, 2, 2, 3, 4 and 4 splits, the last ones uneven
    sizes = [1, 129, 3, 40, 5, 128, 17, 2047, 2049, 4097, 2000]
    edges = {1: [8], 2: [9], 3: [8, 9], 4: [10], 5: [8, 10], 6: [8, 9, 10], 7: [8, 9, 10, 11]}
    X, gb = _check(ctx, oracle, sizes, edges, d, k, "splits")
    ids, dist, _ = ctx.group_knn([int(gb[8])], [sizes[7]], 32)
    _assert_rows_equal(ids, dist, None, *oracle.intra_exact(X, int(gb[8]), sizes[7], 32), None, f"lists d={d}")


@pytest.mark.parametrize("n_child", [1, 63, 64, 65, 511, 512, 513, 1100])
def test_item_counts(ctx, oracle, n_child):
    # one item a child group (9 rows, a union of 300: one split), then one of a single tile
    sizes = [9] * n_child + [140, 300]
    edges = {g: [n_child + 2] for g in range(1, n_child + 1)}
    _check(ctx, oracle, sizes, edges, 450, 6, f"{n_child} items")
