"""The pinned memory of host calls is bounded: inputs above 8 MB are copied
from where they are, large batches' results come in pieces, and both answer as
smaller calls do."""
import numpy as np
import pytest

from tests.helpers import need_gpu, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    need_gpu()
    from browservec_amd import DeviceContext

    c = DeviceContext(0)
    yield c
    c.destroy()


def mapped():
    """Bytes of device and pinned host memory mapped into the process."""
    size = 0
    with open("/proc/self/maps") as f:
        for line in f:
            part = line.split()
            if part[1].startswith("rw") and len(part) > 5 and part[5].startswith("/dev/dri/render"):
                lo, hi = part[0].split("-")
                size += int(hi, 16) - int(lo, 16)
    return size


def test_a_long_row_list_leaves_no_pinned_copy(ctx):
    """24 million listed rows (96 MB), each row often, against the list's
    distinct rows: on the device the list and as many order words, and no
    pinned copy besides."""
    from browservec_amd import FlatIndex

    n, dim, k = 3000, 16, 9
    say("long row list")
    rng = np.random.default_rng(1)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    idx = FlatIndex(ctx, dim, "l2")
    idx.append(x, n)
    q = rng.standard_normal(dim).astype(np.float32)
    once = rng.permutation(n)[:2500].astype(np.uint32)
    short = idx.query_rows(q, once, k)
    many = np.resize(once, 24_000_000)  # (9,600 times each: the best row fills the answer)
    before = mapped()
    hits = idx.query_rows(q, many, k)
    grown = mapped() - before
    assert [(h.row, h.score) for h in hits] == [(short[0].row, short[0].score)] * k
    assert grown < 2.5 * many.nbytes, grown
    idx.destroy()


@pytest.mark.parametrize("nq,k", [(12_000, 100), (3, 1)])
def test_graph_results_in_pieces(ctx, nq, k):
    """12,000 queries x 100 hits (9.6 MB of results) in one call equal the same
    queries in small ones."""
    from browservec_amd.index import GraphSearcher

    n, dim, degree = 4000, 8, 8
    say("graph pieces", nq, k)
    rng = np.random.default_rng(2)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    g = GraphSearcher(ctx, dim, "l2", degree)
    g.append(x, n)
    g.upload_graph(rng.integers(0, n, (n, degree)).astype(np.uint32), n)
    q = rng.standard_normal((nq, dim)).astype(np.float32)
    rows, scores, cnt = g.search_arrays(q, nq, k, 128, 0)
    for s in range(0, nq, 4001):
        m = min(4001, nq - s)
        r, sc, c = g.search_arrays(q[s:s + m], m, k, 128, 0)
        assert np.array_equal(rows[s:s + m], r) and np.array_equal(cnt[s:s + m], c)
        assert np.array_equal(scores[s:s + m].view(np.uint32), sc.view(np.uint32))
    g.destroy()


def test_large_query_batches(ctx):
    """1,024 host queries of 2,304 dimensions (9.4 MB) and a mask, against one
    query at a time."""
    from browservec_amd import FlatIndex

    n, dim, nq, k = 700, 2304, 1024, 5
    say("large host batch")
    rng = np.random.default_rng(3)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    idx = FlatIndex(ctx, dim, "dot")
    idx.append(x, n)
    q = rng.standard_normal((nq, dim)).astype(np.float32)
    rows, scores, cnt = idx.search(q, 0, k)
    for i in (0, 511, nq - 1):
        r, s, c = idx.search(q[i:i + 1], 0, k)
        assert np.array_equal(rows[i], r[0]) and cnt[i] == c[0] == k
        assert np.array_equal(scores[i].view(np.uint32), s[0].view(np.uint32))
    idx.destroy()
