"""GPU parity of the item order of long operand rows (d > 448): runs of 64 consecutive items
per XCD with take-over at the end of the list, and cross unions cut into up to 4 splits of at
least 2048 candidates.  Either side of the row width, of each split count and of the rules that
take them, item counts below, at and past a round of 8 runs, short and long queues.  Rows bit
for bit against the CPU oracle."""
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


@pytest.mark.parametrize("n_child", [1, 63, 64, 65, 511, 512, 513, 1100, 8187, 8188, 8191, 8699, 9300])
def test_item_counts(ctx, oracle, n_child):
    # one item a child group (9 rows, a union of 300: three tiles), then four items of a single
    # tile; runs are taken from 8192 items on, a round of 8 runs is 512
    sizes = [9] * n_child + [400, 300, 100]
    edges = {g: [n_child + 2] for g in range(1, n_child + 1)}
    edges[n_child + 1] = [n_child + 3]
    _check(ctx, oracle, sizes, edges, 450, 6, f"{n_child} items")


@pytest.mark.parametrize("n,k", [(4200, 6), (8193, 32), (9000, 63)])
def test_long_lists(ctx, oracle, n, k):
    # groups above 4096 points: runs of their query blocks (33, 65 and 71 items)
    print(f"runs lists n={n} k={k}", flush=True)
    X = np.random.default_rng(n).standard_normal((n, 450)).astype(np.float32)
    ctx.prepare_vectors(X)
    ids, dist, _ = ctx.group_knn([0], [n], k)
    _assert_rows_equal(ids, dist, None, *oracle.intra_exact(X, 0, n, k), None, f"lists n={n}")


@pytest.mark.parametrize("d,n_child,k,splits", [
    (512, 1300, 6, 4), (512, 1300, 7, 3), (512, 1300, 8, 3), (512, 1300, 9, 1), (512, 1300, 40, 1),  # even
    (512, 100, 6, 4), (512, 100, 8, 4), (512, 100, 9, 4), (512, 100, 40, 4),                          # few long items
    (448, 100, 9, 1), (448, 1300, 6, 1)])
def test_split_rule(ctx, d, n_child, k, splits):
    """Unions of 8192 candidates: how many splits they get (a long queue or an even plan at k >= 9
    only lost by them), the rows the same as a plan of the other number of splits gives."""
    print(f"split rule d={d} n={n_child} k={k}", flush=True)
    sizes = [10] * n_child + [8192]
    gb = np.concatenate([[0, 0], np.cumsum(sizes)]).astype(np.uint32)
    op = np.minimum(np.maximum(np.arange(n_child + 3) - 1, 0), n_child).astype(np.uint32)
    oi = np.full(n_child, n_child + 1, np.uint32)
    X = np.random.default_rng(k).standard_normal((int(gb[-1]), d)).astype(np.float32)
    ctx.prepare_vectors(X)
    ids, dist, size, st = ctx.cross_topk(gb, op, oi, k)
    assert st["work_items"] == splits * n_child
    few = np.minimum(op, 20).astype(np.uint32)  # the first 20 groups alone: few long items
    ids2, dist2, size2, _ = ctx.cross_topk(gb, few, oi[:20], k)
    _assert_rows_equal(ids[:200], dist[:200], size[:200], ids2[:200], dist2[:200], size2[:200], f"d={d} k={k}")
