"""GPU tests of calls that find no device memory for their buffers while the half base set is
allocated (UNG_HIP_SHORT_WITH_HALF=1 refuses every growth until then): it is freed and the call
runs on the split operands, its rows the same as an ordinary context's.  Each entry point that
grows buffers, the group call in flight among them."""
import ctypes as C
import os

import numpy as np
import pytest

import filtervectorcode_refactor_amd as F

pytestmark = pytest.mark.gpu


def _ctx(name):
    os.environ[name] = "1"
    try:
        return F.HipContext(0)
    finally:
        del os.environ[name]


@pytest.fixture(scope="module")
def plain():
    c = F.HipContext(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def split():
    c = _ctx("UNG_HIP_NO_HALF")
    yield c
    c.close()


@pytest.fixture
def short():
    c = _ctx("UNG_HIP_SHORT_WITH_HALF")
    yield c
    c.close()


SIZES = [1, 130, 300, 4300, 700]
GB = np.concatenate([[0, 0], np.cumsum(SIZES)]).astype(np.uint32)
OP, OI = np.array([0, 0, 2, 3, 5, 5, 5], np.uint32), np.array([4, 5, 4, 4, 5], np.uint32)
BEGIN, SIZE = GB[[2, 4]], np.array([SIZES[1], SIZES[3]], np.uint32)


def _x(d):
    return np.random.default_rng(d).standard_normal((int(GB[-1]), d)).astype(np.float32)


def _same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))


@pytest.mark.parametrize("d", [40, 512])
def test_cross(plain, split, short, d):
    print(f"short of memory: cross d={d}", flush=True)
    for c in (plain, split, short):
        c.prepare_vectors(_x(d))
    *want, _ = plain.cross_topk(GB, OP, OI, 6)
    st2 = split.cross_topk(GB, OP, OI, 6)[3]
    *got, st = short.cross_topk(GB, OP, OI, 6)
    _same(got, want)
    for f in ("select_bytes", "work_items", "rows", "pairs", "select_launches"):
        assert st[f] == st2[f], f
    _same(short.cross_topk(GB, OP, OI, 40)[:3], plain.cross_topk(GB, OP, OI, 40)[:3])


def test_lists_and_prune(plain, split, short):
    print("short of memory: lists", flush=True)
    for c in (plain, split, short):
        c.prepare_vectors(_x(96))
    *want, _ = plain.group_knn(BEGIN, SIZE, 32)
    st2 = split.group_knn(BEGIN, SIZE, 32)[2]
    *got, st = short.group_knn(BEGIN, SIZE, 32)
    _same(got, want)
    assert st["select_bytes"] == st2["select_bytes"] and st["select_launches"] == 1
    # buffers of the lists are there now: the half set stays until the packed rows, then the prune
    short.prepare_vectors(_x(96))
    assert short.group_knn(BEGIN, SIZE, 32)[2]["select_bytes"] < st2["select_bytes"]
    _same(short.pack_anchor_rows(None, None, 64, 32, 24)[:2], plain.pack_anchor_rows(None, None, 64, 32, 24)[:2])
    assert short.group_knn(BEGIN, SIZE, 32)[2]["select_bytes"] == st2["select_bytes"]
    short.prepare_vectors(_x(96))
    assert short.group_knn(BEGIN, SIZE, 32)[2]["select_bytes"] < st2["select_bytes"]
    _same(short.prune_group_graph(None, None, 32, 32, 32, 1.2)[:2], plain.prune_group_graph(None, None, 32, 32, 32, 1.2)[:2])
    assert short.group_knn(BEGIN, SIZE, 32)[2]["select_bytes"] == st2["select_bytes"]


def test_overlapped_calls(plain, split, short):
    """Refused in begin; then, its buffers there, in the additional edges while the lists run."""
    print("short of memory: overlapped", flush=True)
    for c in (plain, split, short):
        c.prepare_vectors(_x(96))

    def run(c):
        st = c.cross_intra_begin(GB, OP, OI, 6, BEGIN, SIZE, 32)
        ep, ef, et, _ = c.additional_edges(GB, OP, OI, 6)
        st2 = c.intra_end()
        ids, dist, size, _ = c.download_cross()
        lids, ldist, _ = c.download_group()
        return (ids, dist, size, lids, ldist, ep, ef, et), st["select_bytes"], st2["select_bytes"]

    want, *half = run(plain)
    _, *full = run(split)
    got, *b = run(short)
    _same(got, want)
    assert b == full and half != full
    fresh = _ctx("UNG_HIP_SHORT_WITH_HALF")
    fresh.prepare_vectors(_x(96))
    fresh.cross_intra_begin(GB, OP, OI, 16, BEGIN, SIZE, 40)  # (split rows as long as the half ones below)
    fresh.intra_end()
    fresh.prepare_vectors(_x(96))  # the half set again; no buffers of the additional edges yet
    got, *b = run(fresh)
    _same(got, want)
    assert b == half
    assert fresh.cross_topk_device(GB, OP, OI, 6)["select_bytes"] == full[0]
    fresh.close()


def test_half_set_freed_where_unusable():
    """No copy is kept of a base set outside the half operands' range."""
    hip = C.CDLL("libamdhip64.so")
    n, d = 400_000, 256
    c = F.HipContext(0)
    x = np.ones((n, d), np.float32)
    free = []
    for v in (1.0, 1e20):
        x[0, 0] = v
        c.prepare_vectors(x)
        m, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(m), C.byref(total)) == 0
        free.append(m.value)
    c.close()
    assert free[1] - free[0] >= n * d * 2 * 0.9
