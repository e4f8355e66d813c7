"""GPU tests of calls whose half pre-selection cannot certify its rows (data off the origin:
the operands' rounding error grows with the vectors' norms, their distances do not).  Such a
call is repeated on the split operands.  Every entry point, the register-query layout and the
restaged panels; rows bit for bit against the CPU oracle, or against a context that has the
split operands alone; the statistics count both selects.  The half select gives up soon: past
a count of rows it knows it will not certify it runs no further item, and no merge."""
import ctypes as C
import os

import numpy as np
import pytest

import filtervectorcode_refactor_amd as F
from test_gpu_parity import _assert_rows_equal
from test_zz_no_alloc import DeviceRows

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = F.HipContext(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def split_ctx():
    old = os.environ.get("UNG_HIP_NO_HALF")
    os.environ["UNG_HIP_NO_HALF"] = "1"
    try:
        c = F.HipContext(0)
    finally:
        if old is None:
            del os.environ["UNG_HIP_NO_HALF"]
        else:
            os.environ["UNG_HIP_NO_HALF"] = old
    yield c
    c.close()


def _far(n, d, norm, sigma, seed):
    rng = np.random.default_rng(seed)
    c = rng.standard_normal(d)
    return (sigma * rng.standard_normal((n, d)) + norm * c / np.linalg.norm(c)).astype(np.float32)


SIZES = [1, 130, 300, 2100, 700]  # three child groups, two target groups
GB = np.concatenate([[0, 0], np.cumsum(SIZES)]).astype(np.uint32)
OP, OI = np.array([0, 0, 2, 3, 5, 5, 5], np.uint32), np.array([4, 5, 4, 4, 5], np.uint32)


# norms at which the half operands leave nearly every row uncertified, the split ones few
FAR = [(128, 30, 6), (128, 30, 12), (128, 30, 40), (100, 30, 6), (200, 45, 6), (512, 45, 6), (512, 45, 12), (512, 30, 40)]


@pytest.mark.parametrize("d,norm,k", FAR)
def test_cross(ctx, split_ctx, oracle, d, norm, k):
    print(f"retry cross d={d} k={k}", flush=True)
    X = _far(int(GB[-1]), d, norm, 0.3, d + k)
    ctx.prepare_vectors(X)
    ids, dist, size, st = ctx.cross_topk(GB, OP, OI, k)
    assert st["select_launches"] == 2 and st["fallback_rows"] < 100
    split_ctx.prepare_vectors(X)
    st2 = split_ctx.cross_topk(GB, OP, OI, k)[3]
    assert st["select_bytes"] > st2["select_bytes"] and st["padded_pairs"] > st2["padded_pairs"]
    ip, ii = F.in_neighbors(OP, OI)
    _assert_rows_equal(ids, dist, size, *oracle.cross_exact(X, GB, ip, ii, k), f"d={d} k={k}")


@pytest.mark.parametrize("d,norm,k", [(128, 30, 6), (512, 45, 6)])
def test_overlapped_calls(ctx, oracle, d, norm, k):
    """Cross edges and lists both repeated, the additional edges between them."""
    print(f"retry overlapped d={d}", flush=True)
    X = _far(int(GB[-1]), d, norm, 0.3, 3 * d)
    ctx.prepare_vectors(X)
    begin, size = GB[[2, 4, 5]], np.array([SIZES[1], SIZES[3], SIZES[4]], np.uint32)
    st = ctx.cross_intra_begin(GB, OP, OI, k, begin, size, 32)
    ep, ef, et, _ = ctx.additional_edges(GB, OP, OI, k)
    st2 = ctx.intra_end()
    assert st["select_launches"] == 2 and st2["select_launches"] == 2
    ids, dist, _, _ = ctx.download_cross()
    ip, ii = F.in_neighbors(OP, OI)
    oi, od, _ = oracle.cross_exact(X, GB, ip, ii, k)
    _assert_rows_equal(ids, dist, None, oi, od, None, f"d={d}")
    oep, oef, oet = oracle.additional_edges(X, GB, OP, OI, oi, k)
    assert np.array_equal(ep, oep) and np.array_equal(ef, oef) and np.array_equal(et, oet)
    lids, ldist, _ = ctx.download_group()
    row = 0
    for b, n in zip(begin.tolist(), size.tolist()):
        ri, rd = oracle.intra_exact(X, b, n, 32)
        _assert_rows_equal(lids[row:row + n], ldist[row:row + n], None, ri, rd, None, f"lists d={d} n={n}")
        row += n


def _noalloc(ctx, n, k, *graph):
    rows = DeviceRows(C.CDLL("libamdhip64.so"), n, k)
    try:
        st = ctx.cross_topk_noalloc(*graph, k, *rows.addrs())
        return *rows.download(), st
    finally:
        rows.free()


@pytest.mark.parametrize("d,norm,k", [(128, 30, 6), (128, 30, 40), (512, 45, 12)])
def test_noalloc(ctx, oracle, d, norm, k):
    print(f"retry noalloc d={d} k={k}", flush=True)
    X = _far(int(GB[-1]), d, norm, 0.3, 5 * d + k)
    ctx.prepare_vectors(X)
    ids, dist, size, st = _noalloc(ctx, X.shape[0], k, GB, OP, OI)
    assert st["select_launches"] == 2 and st["allocations"] == 0
    ip, ii = F.in_neighbors(OP, OI)
    _assert_rows_equal(ids, dist, size, *oracle.cross_exact(X, GB, ip, ii, k), f"noalloc d={d} k={k}")


def test_noalloc_split_rows_only(ctx, split_ctx):
    """520k rows: the scratch holds partial rows of 10 entries (split operands), not of 16."""
    sizes = [200_000, 200_000, 120_000, 140]
    gb = np.concatenate([[0, 0], np.cumsum(sizes)]).astype(np.uint32)
    op, oi = np.array([0, 0, 1, 2, 3, 3], np.uint32), np.array([4, 4, 4], np.uint32)
    X = np.random.default_rng(77).standard_normal((int(gb[-1]), 8)).astype(np.float32)
    ctx.prepare_vectors(X)
    split_ctx.prepare_vectors(X)
    ids, dist, size, st = _noalloc(ctx, X.shape[0], 6, gb, op, oi)
    wi, wd, ws, st2 = split_ctx.cross_topk(gb, op, oi, 6)
    assert st["select_launches"] == 1 and st["select_bytes"] == st2["select_bytes"]
    _assert_rows_equal(ids, dist, size, wi, wd, ws, "noalloc on split rows")


def _check_cross_gives_up(ctx, split_ctx, X, gb, op, oi, k, what):
    ctx.prepare_vectors(X)
    split_ctx.prepare_vectors(X)
    ids, dist, size, st = ctx.cross_topk(gb, op, oi, k)
    wi, wd, ws, st2 = split_ctx.cross_topk(gb, op, oi, k)
    _assert_rows_equal(ids, dist, size, wi, wd, ws, what)
    assert st["select_launches"] == 2 and st2["select_launches"] == 1
    # the items in flight when it gives up (at most 512 blocks), of 2,000 or 900
    assert st2["padded_pairs"] < st["padded_pairs"] < 1.6 * st2["padded_pairs"]
    assert st["select_bytes"] > st2["select_bytes"]


@pytest.mark.parametrize("d,k", [(100, 6), (200, 6), (128, 12), (200, 32)])
def test_cross_gives_up(ctx, split_ctx, d, k):
    print(f"give up cross d={d} k={k}", flush=True)
    sizes = [64] * 2000 + [1000]
    gb = np.concatenate([[0, 0], np.cumsum(sizes)]).astype(np.uint32)
    op = np.minimum(np.maximum(np.arange(2003) - 1, 0), 2000).astype(np.uint32)
    oi = np.full(2000, 2001, np.uint32)
    X = _far(int(gb[-1]), d, 20 if k == 6 else 12, 0.1, d + k)
    _check_cross_gives_up(ctx, split_ctx, X, gb, op, oi, k, f"d={d} k={k}")


def test_cross_gives_up_on_split_rows(ctx, split_ctx):
    """300 unions of 70,000 candidates, three splits each."""
    print("give up split rows", flush=True)
    sizes = [128] * 300 + [70_000]
    gb = np.concatenate([[0, 0], np.cumsum(sizes)]).astype(np.uint32)
    op = np.minimum(np.maximum(np.arange(303) - 1, 0), 300).astype(np.uint32)
    X = _far(int(gb[-1]), 128, 12, 0.1, 9)
    _check_cross_gives_up(ctx, split_ctx, X, gb, op, np.full(300, 301, np.uint32), 12, "split rows")


@pytest.mark.parametrize("d,k", [(64, 32), (128, 32), (200, 32), (200, 63)])
def test_lists_give_up(ctx, split_ctx, d, k):
    """2,100 items of 300-point groups: the filter-and-buffer select (d <= 128) and the register
    queues."""
    print(f"give up lists d={d} k={k}", flush=True)
    size = np.full(700, 300, np.uint32)
    begin = np.arange(700, dtype=np.uint32) * 300
    X = _far(210_000, d, 12, 0.1, d)
    ctx.prepare_vectors(X)
    split_ctx.prepare_vectors(X)
    ids, dist, st = ctx.group_knn(begin, size, k)
    wi, wd, st2 = split_ctx.group_knn(begin, size, k)
    _assert_rows_equal(ids, dist, None, wi, wd, None, f"lists d={d} k={k}")
    assert st["select_launches"] == 2 and st2["select_launches"] == 1
    assert st["padded_pairs"] < 1.6 * st2["padded_pairs"]
