"""GPU tests of the bf16 prefilter of fp32 query batches: batches return the
rows and score bits of single queries at every edge of its tiles (32 rows, 128
dimensions, 16-byte pieces, 256 or 128 queries), and rows and queries that its
bounds say nothing about are kept."""
import numpy as np
import pytest

from tests.helpers import need_gpu, say

pytestmark = pytest.mark.gpu

SAMPLE = 16384  # rows of the batch passes' sample


@pytest.fixture(scope="module")
def ctx():
    need_gpu()
    from browservec_amd import DeviceContext

    c = DeviceContext(0)
    yield c
    c.destroy()


def same_as_singles(idx, qs, k, which):
    batch = idx.query_batch(qs, len(qs), k)
    # (the prefilter's passes scan a sample besides the rows)
    assert idx.stats()["last_scanned_rows"] > (idx.size + SAMPLE) * len(qs)
    for i in which:
        one = idx.query(qs[i], k)
        assert [h.row for h in batch[i]] == [h.row for h in one], i
        a = np.float32([h.score for h in batch[i]]).view(np.uint32)
        assert np.array_equal(a, np.float32([h.score for h in one]).view(np.uint32)), i


@pytest.mark.parametrize("metric,dim,n,nq", [
    ("cosine", 5, 1_000_000, 300), ("l2", 31, 200_001, 257), ("cosine", 127, 60_000, 300),
    ("l2", 129, 60_033, 300), ("dot", 300, 40_000, 256), ("cosine", 383, 16_385, 300),
    ("l2", 514, 20_000, 300), ("cosine", 767, 20_001, 260), ("l2", 768, 20_031, 300),
    ("dot", 769, 20_000, 129), ("cosine", 1001, 20_000, 300), ("l2", 1024, 16_400, 130),
])
def test_batches_equal_singles(ctx, metric, dim, n, nq):
    from browservec_amd import FlatIndex

    say("bf16 prefilter", metric, dim, n, nq)
    rng = np.random.default_rng(dim)
    data = rng.standard_normal((n, dim), dtype=np.float32)
    data *= rng.uniform(0.5, 2.0, (n, 1)).astype(np.float32)
    idx = FlatIndex(ctx, dim, metric)
    idx.append(data[: n // 3], n // 3)
    idx.append(data[n // 3:], n - n // 3)
    qs = (data[rng.integers(0, n, nq)] + 0.3 * rng.standard_normal((nq, dim))).astype(np.float32)
    same_as_singles(idx, qs, 10, (0, 31, 32, 127, 128, nq // 2, nq - 1))
    idx.destroy()


@pytest.mark.parametrize("metric", ["dot", "l2"])
def test_rows_and_queries_without_bounds(ctx, metric):
    """Rows and queries whose squares or products leave the range of f32, that
    are not finite, zero or subnormal; 1001 dimensions, so that a row's last
    piece also holds elements of the next row."""
    from browservec_amd import FlatIndex

    dim, n, nq = 1001, 17_000, 140
    say("bf16 prefilter out of range", metric)
    rng = np.random.default_rng(9)
    data = rng.standard_normal((n, dim), dtype=np.float32)
    data[5] = 0
    data[6] *= np.float32(1e-42)
    data[7] *= np.float32(1e-20)
    data[100, 3] = np.inf
    data[101, 0] = -np.inf
    data[8000, 1000] = np.float32(3e38)
    data[9000, 0] = np.nan
    data[16_999, 7] = np.float32(2e19)
    idx = FlatIndex(ctx, dim, metric)
    idx.append(data, n)
    qs = rng.standard_normal((nq, dim), dtype=np.float32)
    qs[1] = 0
    qs[2] *= np.float32(1e-42)
    qs[3] *= np.float32(1e-20)
    qs[4, 9] = np.float32(3e38)
    qs[5, 0] = np.inf
    qs[6] *= np.float32(1e18)
    same_as_singles(idx, qs, 10, range(8))
    idx.destroy()


def test_large_k_batches_bound_their_scratch(ctx):
    """1,024 queries at k 1000 over 1M rows keep up to 250,000 rows each: the
    batch runs in passes whose scratch stays near 3 GiB (10 in one), and
    every pass answers as single queries do."""
    import torch

    from browservec_amd import FlatIndex

    dim, n, nq, k = 8, 1_000_000, 1024, 1000
    say("bf16 prefilter scratch", nq, k)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(n, dim, generator=g, device="cuda")
    q = torch.randn(nq, dim, generator=g, device="cuda")
    torch.cuda.synchronize()
    idx = FlatIndex(ctx, dim, "l2")
    idx.append_device(x.data_ptr(), n)
    rows = torch.zeros(nq, k, dtype=torch.int32, device="cuda")
    scores = torch.zeros(nq, k, device="cuda")
    cnt = torch.zeros(nq, dtype=torch.int32, device="cuda")
    idx.sync()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    idx.search_device(q.data_ptr(), nq, 0, k, rows.data_ptr(), scores.data_ptr(), cnt.data_ptr())
    idx.sync()
    assert free - torch.cuda.mem_get_info()[0] < 5 << 30
    for i in (0, 255, 256, 700, nq - 1):
        r, s, c = idx.search(q[i:i + 1].cpu().numpy(), 0, k)
        assert c[0] == cnt[i].item() == k
        assert np.array_equal(r[0], rows[i].cpu().numpy().view(np.uint32)), i
        assert np.array_equal(s[0].view(np.uint32), scores[i].cpu().numpy().view(np.uint32)), i
    idx.destroy()


def device_rows(idx, q, nq, k, width):
    import torch

    rows = torch.zeros(nq, k, dtype=torch.int32, device="cuda")
    scores = torch.zeros(nq, k, device="cuda")
    cnt = torch.zeros(nq, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for i in range(0, nq, width):
        idx.search_device(q[i:].data_ptr(), width, 0, k, rows[i:].data_ptr(), scores[i:].data_ptr(), cnt[i:].data_ptr())
    idx.sync()
    return rows.cpu().numpy(), scores.cpu().numpy().view(np.uint32), cnt.cpu().numpy()


def equals_fused(idx, q, nq, k):
    """A batch against the fused scan of each query alone (which calls on two
    query streams run); returns the rows the batch scanned."""
    a = device_rows(idx, q, nq, k, nq)
    scanned = idx.stats()["last_scanned_rows"]
    idx.set_query_streams(2)
    b = device_rows(idx, q, nq, k, 1)
    idx.set_query_streams(1)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    return scanned


@pytest.mark.parametrize("metric,dim,n,size,nq", [("cosine", 96, 150_000, 200, 256), ("l2", 768, 60_000, 200, 200),
                                                  ("dot", 1000, 40_000, 3000, 130)])
def test_neighbouring_rows_of_a_corpus_in_topic_order(ctx, metric, dim, n, size, nq):
    """Whole tiles of a topic pass for every query of a wave, more than its
    staging buffer holds: the rest go through the queries' spill lists, and no
    query needs a scan of its own (what was scanned is the sample, the rows
    and the kept rows)."""
    import torch

    from browservec_amd import FlatIndex

    say("topic order", metric, dim, n, size, nq)
    g = torch.Generator(device="cuda").manual_seed(dim)
    centres = torch.nn.functional.normalize(torch.randn(n // size + 1, dim, generator=g, device="cuda"), dim=1)
    x = centres[torch.arange(n, device="cuda") // size] + torch.randn(n, dim, generator=g, device="cuda") * 2 / dim ** 0.5
    if metric == "cosine":
        x = torch.nn.functional.normalize(x, dim=1).contiguous()
    torch.cuda.synchronize()
    idx = FlatIndex(ctx, dim, metric)
    idx.append_device(x.data_ptr(), n)
    s = n // 2 // size * size + size // 3
    scanned = equals_fused(idx, x[s:s + nq].contiguous(), nq, 10)
    assert (n + SAMPLE) * nq < scanned < (n + SAMPLE) * nq + nq * 2 * size + 8 * n
    idx.destroy()


@pytest.mark.parametrize("metric,dim,products", [("dot", 768, True), ("l2", 128, True), ("dot", 100, False)])
def test_rows_with_a_large_part_in_common(ctx, metric, dim, products):
    """A common mean keeps every row under the bf16 bounds: the batch is run
    again with fp32 products where the dimension has them, else by slot scans,
    and answers as single queries do."""
    import torch

    from browservec_amd import FlatIndex

    n, nq = 60_000, 300
    say("common mean", metric, dim)
    g = torch.Generator(device="cuda").manual_seed(dim)
    mean = 100 if metric == "dot" else 10
    x = torch.randn(n, dim, generator=g, device="cuda") / dim ** 0.5
    x += mean * torch.nn.functional.normalize(torch.randn(dim, generator=g, device="cuda"), dim=0)
    q = x[torch.randint(0, n, (nq,), generator=g, device="cuda")]
    q = (q + 0.1 * torch.randn(nq, dim, generator=g, device="cuda") / dim ** 0.5).contiguous()
    torch.cuda.synchronize()
    idx = FlatIndex(ctx, dim, metric)
    idx.append_device(x.data_ptr(), n)
    scanned = equals_fused(idx, q, nq, 10)
    first = (n + SAMPLE) * nq
    if products:  # (and few rows kept)
        assert 2 * first < scanned < 2 * first + nq * 4000
    else:
        assert scanned == first + n * nq
    idx.destroy()


def test_only_overflowed_queries_are_run_again(ctx):
    """Three kinds of queries in turn: close to the first are rows 1e-6 apart
    (their lists overflow under either bound: slot scans), to the second rows
    1e-3 apart (fp32 products tell them apart), and the third need no second
    pass."""
    import torch

    from browservec_amd import FlatIndex

    dim, n, nq = 64, 80_000, 150
    say("overflow of some")
    g = torch.Generator(device="cuda").manual_seed(8)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    u, v = torch.linalg.qr(rand(dim, 2)).Q.T
    i = torch.arange(n, device="cuda")
    x = torch.nn.functional.normalize(rand(n, dim), dim=1)
    near_u = (i % 8 == 0) | (i % 4 == 1)  # (the sample takes every fourth row)
    near_v = i % 4 >= 2
    x[near_u] = u * (1 + 1e-3 * rand(int(near_u.sum()), 1)) + 1e-3 * rand(int(near_u.sum()), dim) / 8
    x[near_v] = v + 1e-6 * rand(int(near_v.sum()), dim) / 8
    q = rand(nq, dim)
    q -= torch.outer(q @ u, u) + torch.outer(q @ v, v)
    q = torch.nn.functional.normalize(q, dim=1)
    q[0::3] = v + 0.01 * rand(50, dim) / 8
    q[1::3] = u + 0.01 * rand(50, dim) / 8
    q = q.contiguous()
    torch.cuda.synchronize()
    idx = FlatIndex(ctx, dim, "dot")
    idx.append_device(x.contiguous().data_ptr(), n)
    scanned = equals_fused(idx, q, nq, 10)
    least = (n + SAMPLE) * nq + (n + SAMPLE) * 100 + n * 50
    assert least < scanned < least + 50 * SAMPLE * 2 + nq * 4000
    idx.destroy()


def test_a_spill_list_filled_to_its_end(ctx):
    """All rows close to the queries lie in one workgroup's tiles, and one wave
    fills the queries' spill lists with the first 512 of them to the last
    entry; the closest rows lie in the tiles after those."""
    import torch

    from browservec_amd import FlatIndex

    n, dim, nq, k = 5_000_000, 4, 64, 10
    say("spill list full")
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(n, dim, generator=g, device="cuda") * 0.1
    x[:, 0] = -1
    wgs = ctx.info()["cu_count"] // 8 * 8  # one query block: every workgroup of the device
    first = n // 8 // 32 * 32  # (the rows after the first eighth are a pass)
    tile = torch.arange((n - first) // 32, device="cuda")
    tile = tile[tile % wgs == 5]
    assert len(tile) > 512
    rows = (first + tile[:, None] * 32 + torch.arange(32, device="cuda")).flatten()
    x[rows] = 0
    x[rows, 0] = 1 + 0.0015 * torch.arange(len(rows), device="cuda") / len(rows)
    q = torch.zeros(nq, dim, device="cuda")
    q[:, 0] = 1
    torch.cuda.synchronize()
    idx = FlatIndex(ctx, dim, "dot")
    idx.append_device(x.data_ptr(), n)
    equals_fused(idx, q, nq, k)
    best = idx.search(q[:1].cpu().numpy(), 0, k)[0][0]
    assert (best > rows[512 * 32].item()).all()
    idx.destroy()
