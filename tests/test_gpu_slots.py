"""Small batches and short scans (scan_slots + pick_topk) against the fused
single-query scan, which single queries kept on two streams run: the same
arithmetic row by row, so rows, score bits and counts must be identical.
Sizes sit at the edges of a slot, of a wave step and of the selection's list;
rows that tie and masks that leave little are among them."""

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


def make(ctx, kind, dim, n, seed):
    import torch

    from browservec_amd import FlatIndex, QuantIndex

    g = torch.Generator(device="cuda").manual_seed(seed)
    centres = torch.randn(16, dim, generator=g, device="cuda")
    x = centres[torch.randint(0, 16, (n,), generator=g, device="cuda")] * 0.3
    x += torch.randn(n, dim, generator=g, device="cuda")
    if kind != "l2":
        x /= x.norm(dim=1, keepdim=True)
    if kind in ("cosine", "l2"):
        idx = FlatIndex(ctx, dim, kind)
    else:
        idx = QuantIndex(ctx, dim, bits=int(kind[0]), scorer=kind[1:] or "asym")
    torch.cuda.synchronize()
    idx.append_device(x.data_ptr(), n)
    q = x[torch.randint(0, n, (64,), generator=g, device="cuda")] + 0.3 * torch.randn(64, dim, generator=g,
                                                                                     device="cuda") / dim ** 0.5
    return idx, x, q.contiguous()


def both_equal(idx, q, nq, fetch, k):
    import torch

    out = []
    for streams, width in ((1, nq), (2, 1)):
        idx.set_query_streams(streams)
        rows = torch.full((nq, k), -1, dtype=torch.int32, device="cuda")
        scores = torch.zeros(nq, k, device="cuda")
        cnt = torch.zeros(nq, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        for i in range(0, nq, width):
            idx.search_device(q[i:].data_ptr(), width, fetch, k, rows[i:].data_ptr(), scores[i:].data_ptr(),
                              cnt[i:].data_ptr())
        idx.sync()
        out.append([rows.cpu().numpy(), scores.cpu().numpy().view(np.uint32), cnt.cpu().numpy()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("kind,dim,n,nq,fetch,k", [
    ("8", 768, 17, 3, 17, 10), ("8", 300, 4097, 5, 40, 10), ("8", 100, 20011, 33, 100, 32),
    ("8", 768, 300_001, 4, 100, 10),          # several parts per slot
    ("4", 1000, 8193, 4, 160, 10), ("4", 96, 65, 2, 64, 64), ("4", 768, 140_000, 7, 160, 10),
    ("1", 384, 20_000, 1, 1024, 10),          # a fetch above the slots: the list is cut on the way
    ("1", 768, 33_000, 6, 320, 10), ("1", 130, 257, 3, 100, 10), ("1", 1024, 600_000, 2, 200, 10),
    ("1hamming", 768, 50_000, 9, 320, 10), ("1hamming", 100, 3000, 2, 1024, 16),
    ("8int8sym", 256, 9000, 3, 64, 8),
    ("cosine", 384, 20_000, 7, 0, 10), ("l2", 300, 10_007, 20, 0, 50), ("cosine", 77, 2049, 64, 0, 1),
    ("l2", 768, 1, 1, 0, 1), ("cosine", 1024, 70_000, 3, 0, 100), ("cosine", 37, 40_000, 4, 0, 1000),
])
def test_slots_equal_the_fused_scan(ctx, kind, dim, n, nq, fetch, k):
    say("slots", kind, dim, n, nq, fetch, k)
    idx, x, q = make(ctx, kind, dim, n, dim + n)
    both_equal(idx, q[:nq].contiguous(), nq, fetch, k)
    idx.destroy()


@pytest.mark.parametrize("kind", ["8", "4", "1", "1hamming", "cosine"])
def test_slots_equal_rows(ctx, kind):
    """Every row alike: all keys tie, and the lowest rows come back in order."""
    import torch

    from browservec_amd import FlatIndex, QuantIndex

    say("slots ties", kind)
    dim, n, k = 256, 30_000, 40
    idx = FlatIndex(ctx, dim, kind) if kind == "cosine" else QuantIndex(ctx, dim, bits=int(kind[0]),
                                                                        scorer=kind[1:] or "asym")
    x = torch.nn.functional.normalize(torch.randn(1, dim, device="cuda"), dim=1).repeat(n, 1).contiguous()
    torch.cuda.synchronize()
    idx.append_device(x.data_ptr(), n)
    rows, _, cnt = idx.search(x[:3].cpu().numpy(), 0, k)
    assert (cnt == k).all() and np.array_equal(rows, np.tile(np.arange(k, dtype=np.uint32), (3, 1)))
    idx.destroy()


@pytest.mark.parametrize("kind,n,keep", [("8", 20_000, 0.3), ("1", 9_000, 0.01), ("cosine", 33_333, 0.0005), ("4", 5000, 0.0)])
def test_slots_masked(ctx, kind, n, keep):
    """Masked queries return the canonical top k of the kept rows' scan scores."""
    say("slots masked", kind, n, keep)
    idx, x, q = make(ctx, kind, 256, n, n)
    rng = np.random.default_rng(n)
    live = rng.random(n) < keep
    mask = np.zeros((n + 31) // 32, np.uint32)
    np.bitwise_or.at(mask, np.nonzero(live)[0] >> 5, np.uint32(1) << (np.nonzero(live)[0] & 31).astype(np.uint32))
    qh = q[0].cpu().numpy()
    hits = idx.query_masked(qh, 25, mask)
    scores = idx.export_scores(qh)
    rows = np.nonzero(live)[0]
    order = rows[np.lexsort((rows, -scores[rows].astype(np.float64)))][:25]
    assert [h.row for h in hits] == order.tolist()
    assert np.array_equal(np.array([h.score for h in hits], np.float32).view(np.uint32), scores[order].view(np.uint32))
    idx.destroy()


@pytest.mark.parametrize("metric,dim,n_list,k", [("cosine", 768, 1, 1), ("l2", 300, 15, 10), ("dot", 37, 17, 17),
                                                 ("cosine", 3, 200, 100), ("l2", 1001, 4097, 1000),
                                                 ("cosine", 96, 140_000, 20)])
def test_listed_rows_equal_dot_row(ctx, metric, dim, n_list, k):
    """Listed rows (a duplicate among them) score Store.dotRow / l2Row bit for
    bit and come back in canonical order."""
    from browservec_amd import FlatIndex
    from oracle import oracle as o

    say("listed rows", metric, dim, n_list, k)
    rng = np.random.default_rng(dim)
    n = max(n_list + 5, 50)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    idx = FlatIndex(ctx, dim, metric)
    idx.append(x, n)
    lst = rng.permutation(n)[:n_list].astype(np.uint32)
    if n_list > 2:
        lst[-1] = lst[0]
    q = rng.standard_normal(dim).astype(np.float32)
    hits = idx.query_rows(q, lst, k)
    s = np.array([o.l2_row(x[r], q) if metric == "l2" else o.dot_row(x[r], q) for r in lst], np.float64).astype(np.float32)
    order = np.lexsort((lst, -s.astype(np.float64)))[:k]
    assert [h.row for h in hits] == lst[order].tolist()
    assert np.array_equal(np.array([h.score for h in hits], np.float32).view(np.uint32), s[order].view(np.uint32))
    idx.destroy()


def test_more_queries_than_a_launch_takes(ctx):
    """70,000 queries over 300 rows in one call: a launch takes up to 65,535,
    and the rest get one of their own."""
    import torch

    n, dim, nq, k = 300, 16, 70_000, 3
    say("slots", nq, "queries")
    idx, x, _ = make(ctx, "cosine", dim, n, 11)
    q = torch.randn(nq, dim, generator=torch.Generator(device="cuda").manual_seed(12), device="cuda")
    out = []
    for width in (nq, 2500):
        rows = torch.full((nq, k), -1, dtype=torch.int32, device="cuda")
        scores = torch.zeros(nq, k, device="cuda")
        cnt = torch.zeros(nq, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        for i in range(0, nq, width):
            idx.search_device(q[i:].data_ptr(), width, 0, k, rows[i:].data_ptr(), scores[i:].data_ptr(),
                              cnt[i:].data_ptr())
        idx.sync()
        out.append([rows.cpu().numpy(), scores.cpu().numpy().view(np.uint32), cnt.cpu().numpy()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    idx.destroy()


@pytest.mark.parametrize("kind,dim,n,nq,fetch", [("8", 768, 20_000, 1, 60), ("1hamming", 256, 30_000, 5, 100),
                                                 ("4", 384, 20_000, 10, 40), ("cosine", 100, 25_000, 3, 0)])
def test_no_room_for_order_words(ctx, kind, dim, n, nq, fetch):
    """Where a slot scan's scratch does not fit, the query takes the path it
    would take without one and answers the same."""
    say("slots out of memory", kind, nq)
    idx, x, q = make(ctx, kind, dim, n, 21)
    qh = q[:nq].cpu().numpy()
    want = idx.search(qh, fetch, 10)
    ctx.debug_inject("slots_oom")
    got = idx.search(qh, fetch, 10)
    for a, b in zip(want, got):
        assert np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))
    idx.destroy()


@pytest.mark.parametrize("kind,n,dim,fetch", [("8", 600_000, 1024, 100), ("8int8sym", 600_000, 1024, 100),
                                              ("4", 2_100_000, 1024, 160), ("8", 600_000, 1024, 300)])
def test_single_queries_over_large_codes(ctx, kind, n, dim, fetch):
    """Single queries on either side of the sizes at which the fused scan takes
    them, against the slot scan of two queries at once."""
    import torch

    say("large single", kind, n, fetch)
    idx, x, q = make(ctx, kind, dim, n, 5)
    del x
    out = []
    for width in (1, 2):
        rows = torch.full((4, 10), -1, dtype=torch.int32, device="cuda")
        scores = torch.zeros(4, 10, device="cuda")
        cnt = torch.zeros(4, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        for i in range(0, 4, width):
            idx.search_device(q[i:].data_ptr(), width, fetch, 10, rows[i:].data_ptr(), scores[i:].data_ptr(),
                              cnt[i:].data_ptr())
        idx.sync()
        out.append([rows.cpu().numpy(), scores.cpu().numpy().view(np.uint32), cnt.cpu().numpy()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    idx.destroy()
    torch.cuda.empty_cache()


@pytest.mark.parametrize("kind,dim,n,nq,fetch,k", [("8", 1000, 3000, 1, 66, 10), ("4", 1024, 5000, 7, 1024, 1024),
                                                   ("1", 768, 40_000, 2, 96, 96), ("1hamming", 1024, 100, 3, 100, 5),
                                                   ("8int8sym", 2048, 9000, 2, 33, 33)])
def test_shared_rerank_equals_the_fused_scan(ctx, kind, dim, n, nq, fetch, k):
    """A re-rank that several workgroups share (65,536 elements and more, up to
    seven queries), fewer sixteens of rows than workgroups among them."""
    say("shared re-rank", kind, dim, n, nq, fetch, k)
    idx, x, q = make(ctx, kind, dim, n, dim + n)
    both_equal(idx, q[:nq].contiguous(), nq, fetch, k)
    both_equal(idx, q[8:8 + nq].contiguous(), nq, fetch, k)  # (the counters are as they were)
    idx.destroy()
