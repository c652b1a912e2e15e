"""Quantized batches on the matrix-core passes, at sizes that go there, against
the fused scan of each query alone (which calls on two query streams run).
A batch that took the pass scanned its sample besides every row, and the rows
again of a query whose kept rows overflowed: stats tell."""

import numpy as np
import pytest

from tests.helpers import need_gpu, say

pytestmark = pytest.mark.gpu

SAMPLE = 16384  # rows of the passes' sample


@pytest.fixture(scope="module")
def ctx():
    need_gpu()
    from browservec_amd import DeviceContext

    c = DeviceContext(0)
    yield c
    c.destroy()


def index_of(ctx, kind, x):
    import torch

    from browservec_amd import QuantIndex

    idx = QuantIndex(ctx, x.shape[1], bits=int(kind[0]), scorer=kind[1:] or "asym")
    torch.cuda.synchronize()
    idx.append_device(x.data_ptr(), x.shape[0])
    return idx


def search(idx, q, which, width, fetch, k):
    import torch

    rows = torch.full((len(q), k), -1, dtype=torch.int32, device="cuda")
    scores = torch.zeros(len(q), k, device="cuda")
    cnt = torch.zeros(len(q), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for i in which:
        idx.search_device(q[i:].data_ptr(), width, fetch, k, rows[i:].data_ptr(), scores[i:].data_ptr(),
                          cnt[i:].data_ptr())
    idx.sync()
    return rows.cpu().numpy(), scores.cpu().numpy().view(np.uint32), cnt.cpu().numpy()


def batch_equals_fused(idx, q, fetch, k):
    """Returns the rows that the batch scanned."""
    nq = len(q)
    batch = search(idx, q, [0], nq, fetch, k)
    scanned = idx.stats()["last_scanned_rows"]
    which = sorted({0, 1, 31, 32, nq // 2, nq - 2, nq - 1, *range(3, nq, max(1, nq // 20))} & set(range(nq)))
    idx.set_query_streams(2)
    alone = search(idx, q, which, 1, fetch, k)
    idx.set_query_streams(1)
    for a, b in zip(batch, alone):
        assert np.array_equal(a[which], b[which])
    return scanned


def mixture(n, dim, nq, seed, topics=50):
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed)
    centres = torch.nn.functional.normalize(torch.randn(topics, dim, generator=g, device="cuda"), dim=1)
    x = centres[torch.randint(0, topics, (n,), generator=g, device="cuda")]
    x = torch.nn.functional.normalize(x + 0.1 * torch.randn(n, dim, generator=g, device="cuda"), dim=1)
    q = x[torch.randint(0, n, (nq,), generator=g, device="cuda")]
    q = torch.nn.functional.normalize(q + 0.05 * torch.randn(nq, dim, generator=g, device="cuda"), dim=1)
    return x.contiguous(), q.contiguous()


@pytest.mark.parametrize("kind,dim,n,nq,fetch,k", [
    ("8", 256, 60_001, 300, 100, 10), ("8", 768, 40_000, 70, 1000, 10), ("8", 100, 200_000, 100, 0, 20),
    ("4", 1000, 40_033, 75, 160, 10), ("4", 256, 60_000, 260, 1000, 1000), ("4", 384, 100_000, 130, 0, 20),
    ("1hamming", 1024, 60_000, 257, 320, 10), ("1hamming", 256, 150_000, 400, 0, 50),
    ("1", 1024, 40_000, 110, 320, 10), ("1", 100, 120_000, 300, 0, 50), ("1", 512, 60_000, 140, 1000, 10),
])
def test_batches_on_the_matrix_cores(ctx, kind, dim, n, nq, fetch, k):
    say("batch route", kind, dim, n, nq, fetch, k)
    x, q = mixture(n, dim, nq, dim + n)
    x[n // 2:n // 2 + 100] = x[:100]  # (rows that tie)
    idx = index_of(ctx, kind, x)
    scanned = batch_equals_fused(idx, q, fetch, k)
    assert (n + SAMPLE) * nq <= scanned < (n + SAMPLE) * nq + n * nq // 2
    idx.destroy()


@pytest.mark.parametrize("kind,dim,n,nq", [("8", 256, 60_000, 200), ("4", 1000, 60_000, 75), ("1hamming", 1024, 80_000, 210),
                                           ("1", 1024, 60_000, 90)])
def test_near_duplicates(ctx, kind, dim, n, nq):
    """Groups of eight rows 1e-4 apart: whole groups lie within the bounds, and
    the exact keys order them."""
    import torch

    say("batch near-duplicates", kind, dim)
    base, q = mixture(n // 8, dim, nq, dim)
    x = base.repeat_interleave(8, 0) + 1e-4 * torch.randn(n, dim, generator=torch.Generator(device="cuda").manual_seed(2),
                                                          device="cuda")
    idx = index_of(ctx, kind, torch.nn.functional.normalize(x, dim=1).contiguous())
    scanned = batch_equals_fused(idx, q, 100, 10)
    assert (n + SAMPLE) * nq <= scanned < (n + SAMPLE) * nq + n * nq // 2
    idx.destroy()


@pytest.mark.parametrize("kind,dim,n,nq", [("8", 256, 60_000, 200), ("4", 1000, 60_000, 75), ("1hamming", 1024, 80_000, 210),
                                           ("1", 1024, 60_000, 90)])
def test_overflow(ctx, kind, dim, n, nq):
    """Three quarters of the rows are one vector, all within every bound of a
    query near it: its list overflows.  Every other 32 queries (a wave's) are
    near it, and only those are run again, together."""
    import torch

    say("batch overflow", kind, dim)
    x, q = mixture(n, dim, nq, dim + 1)
    v = torch.nn.functional.normalize(torch.randn(dim, generator=torch.Generator(device="cuda").manual_seed(3),
                                                  device="cuda"), dim=0)
    x[torch.arange(n, device="cuda") % 4 != 0] = v
    q -= torch.outer(q @ v + 0.5, v)  # (the others away from it)
    near = torch.arange(nq, device="cuda") // 32 % 2 == 1
    q[near] = v + 0.01 * q[near]
    idx = index_of(ctx, kind, x)
    scanned = batch_equals_fused(idx, q.contiguous(), 100, 10)
    least = (n + SAMPLE) * nq + n * int(near.sum())
    assert least <= scanned < least + n * 8
    rows, scores, cnt = idx.search(q.cpu().numpy(), 100, 10)  # (results in pinned memory)
    again = search(idx, q.contiguous(), [0], nq, 100, 10)
    assert np.array_equal(rows.view(np.int32), again[0]) and np.array_equal(scores.view(np.uint32), again[1])
    idx.destroy()


@pytest.mark.parametrize("kind,dim,n,nq,fetch", [("8", 1000, 16_000, 120, 100), ("8", 768, 16_384, 150, 0),
                                                 ("4", 1024, 16_000, 150, 160)])
def test_one_dense_pass(ctx, kind, dim, n, nq, fetch):
    """No more rows than the sample: one dense pass over all of them."""
    say("batch one pass", kind, dim, n)
    x, q = mixture(n, dim, nq, dim + 2)
    idx = index_of(ctx, kind, x)
    assert batch_equals_fused(idx, q, fetch, 10) == n * nq
    idx.destroy()
