"""Performance cases of the search path: what a program that uses the framework
has it do, through its public entry points, over the range of sizes it serves.

A case is a dict of plain values; ``kind`` says which path it takes:

  flat   FlatIndex (fp32): exact top-k of one query or a batch
  quant  QuantIndex (int8, int4, 1-bit asymmetric or Hamming codes): top-`fetch`
         by code score, exact re-rank to top-k, one query or a batch
  ivf    IVFIndex / IVFQuantIndex: probe, scan of the probed lists, top-k
         (quantized kinds: fetch and exact re-rank)
  rows   exact scores of a list of rows (a metadata filter that matched few
         rows) and their top-k
  build  a corpus loaded into an IVF index: append, k-means, lists
  graph  HNSW layer-0 beam search of a batch of queries

``host`` cases go through the calls that take and return host arrays (an
application that holds one query at a time); the others hand over device
buffers (a serving loop that keeps queries and results in HBM).
"""

import functools
import math

import numpy as np
import torch

from browservec_amd import DeviceContext, FlatIndex, QuantIndex
from browservec_amd.index import GraphSearcher, IVFIndex, IVFQuantIndex

SEED = 0x9E3779B9  # the indexes' default rotation seed
CHUNK = 1 << 17
TOPIC = 200  # rows of a graph corpus that share a topic


def listed():
    return [
        # the smallest call: an application with 20,000 embeddings of a small
        # model that asks one question at a time
        dict(name="flat_20k384_q1", kind="flat", n=20_000, dim=384, metric="cosine", nq=1, k=10, host=True),
        # exact search of a large corpus for a batch of queries (ground truth,
        # deduplication, evaluation)
        dict(name="flat_1m768_q256", kind="flat", n=1_000_000, dim=768, metric="cosine", nq=256, k=10, host=False),
        # the headline: one query over a million int8 rows
        dict(name="int8_1m768_q1", kind="quant", bits=8, scorer="asym", n=1_000_000, dim=768, nq=1, fetch=100, k=10,
             host=False),
        # a few users at once, or one question in a few wordings
        dict(name="int8_1m768_q4", kind="quant", bits=8, scorer="asym", n=1_000_000, dim=768, nq=4, fetch=40, k=10,
             host=False),
        # the headline's batch
        dict(name="int8_1m768_q256", kind="quant", bits=8, scorer="asym", n=1_000_000, dim=768, nq=256, fetch=100,
             k=10, host=False),
        # a large int4 corpus, a ragged dimension and row count, a middling
        # batch that is no multiple of a tile
        dict(name="int4_3m1000_q33", kind="quant", bits=4, scorer="asym", n=3_000_017, dim=1000, nq=33, fetch=160,
             k=10, host=False),
        # the most rows per byte: one query over 1-bit codes
        dict(name="bit1_4m1024_q1", kind="quant", bits=1, scorer="asym", n=4_000_000, dim=1024, nq=1, fetch=200, k=10,
             host=False),
        # approximate search of millions of rows, one query: launches and
        # latency more than bytes
        dict(name="ivf8_4m768_q1", kind="ivf", bits=8, n=4_000_000, dim=768, nlist=4096, nprobe=32, nq=1, fetch=40,
             k=10, host=False),
        # the same index under a serving load
        dict(name="ivf8_4m768_q1024", kind="ivf", bits=8, n=4_000_000, dim=768, nlist=4096, nprobe=32, nq=1024,
             fetch=40, k=10, host=False),
        # a metadata filter that matches a few thousand rows (up to 4096 the
        # search scores them exactly, whatever the index)
        dict(name="rows_3000_of_300k768", kind="rows", n=300_000, dim=768, metric="cosine", n_list=3_000, k=10),
        # loading a corpus into an IVF index: the write direction
        dict(name="build_ivf8_500k768", kind="build", bits=8, n=500_000, dim=768, nlist=1024, iters=8),
        # graph search, a small batch
        dict(name="graph_200k768_q64", kind="graph", n=200_000, dim=768, degree=32, nq=64, ef=128, k=10),
    ]


def _logint(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dim(rng):
    """A model's embedding width, or any other."""
    return rng.choice([96, 128, 256, 300, 384, 512, 768, 1000, 1024, rng.randint(64, 1024), rng.randint(64, 1024)])


def draw(rng):
    kind = rng.choice(["flat", "flat", "flat", "quant", "quant", "quant", "quant", "ivf", "ivf", "ivf", "rows",
                       "build", "graph"])
    dim = _dim(rng)
    if kind == "flat":
        n = _logint(rng, 2_000, min(1_000_000, 768_000_000 // dim))
        nq = _logint(rng, 1, 256)
        return dict(kind=kind, n=n, dim=dim, metric=rng.choice(["cosine", "dot", "l2"]), nq=nq,
                    k=_logint(rng, 1, 100), host=nq <= 4 and rng.random() < 0.5)
    if kind == "quant":
        bits = rng.choice([8, 8, 4, 1])
        n = _logint(rng, 5_000, min(4_000_000, 1_500_000_000 // dim))
        nq = max(1, min(_logint(rng, 1, 256), 196_000_000_000 // (n * dim)))
        k = _logint(rng, 1, 32)
        return dict(kind=kind, bits=bits, scorer="hamming" if bits == 1 and dim > 64 and rng.random() < 0.5 else "asym", n=n,
                    dim=dim, nq=nq, fetch=min(1024, k * {8: 4, 4: 16, 1: 32}[bits]), k=k,
                    host=nq <= 4 and rng.random() < 0.5)
    if kind == "ivf":
        bits = rng.choice([8, 8, 4, 1, 0])
        n = _logint(rng, 20_000, min(2_000_000, 1_000_000_000 // dim))
        nlist = _logint(rng, 64, min(4096, n // 100))
        nprobe = _logint(rng, 1, min(64, nlist))
        nq = max(1, min(_logint(rng, 1, 1024), 32_000_000 * nlist // (nprobe * n)))
        k = _logint(rng, 1, 32)
        return dict(kind=kind, bits=bits, n=n, dim=dim, nlist=nlist, nprobe=nprobe, nq=nq,
                    fetch=k * {8: 4, 4: 16, 1: 32, 0: 0}[bits], k=k, host=nq <= 4 and rng.random() < 0.5)
    if kind == "rows":
        n = _logint(rng, 5_000, min(1_000_000, 300_000_000 // dim))
        return dict(kind=kind, n=n, dim=dim, metric=rng.choice(["cosine", "dot", "l2"]),
                    n_list=_logint(rng, 100, min(n, 100_000)), k=_logint(rng, 1, 100))
    if kind == "build":
        n = _logint(rng, 30_000, min(500_000, 384_000_000 // dim))
        return dict(kind=kind, bits=rng.choice([8, 8, 4, 1, 0]), n=n, dim=dim,
                    nlist=_logint(rng, 64, min(1024, n // 100)), iters=rng.randint(3, 10))
    n = _logint(rng, 5_000, 200_000)
    return dict(kind=kind, n=n, dim=min(dim, 768), degree=rng.choice([16, 32, 48]), nq=_logint(rng, 1, 256),
                ef=rng.randint(32, 160), k=rng.randint(1, 20))


# ------------------------------------------------------------------ inputs --
@functools.lru_cache(maxsize=1)
def _context():
    return DeviceContext(0)


def _data(case, seed, nq):
    """Rows of a Gaussian mixture (unit centres, noise of norm 2 to 4 as text
    embeddings spread around their topics; graphs: tight topics that a walk
    can follow) and queries near corpus rows.  cosine: unit rows; dot: lengths
    between 0.5 and 1.5; l2: as they come."""
    n, dim = case["n"], case["dim"]
    metric = case.get("metric", "cosine")
    g = torch.Generator(device="cuda").manual_seed(seed)
    clusters = max(1, min(case.get("nlist", 1024), n // 8))
    if case["kind"] == "graph":
        clusters = -(-n // TOPIC)
    sigma, noise = {"ivf": (0.15, 0.05), "build": (0.15, 0.05), "graph": (0.02, 0.01)}.get(case["kind"], (0.1, 0.05))
    centres = torch.randn(clusters, dim, generator=g, device="cuda")
    centres /= centres.norm(dim=1, keepdim=True)
    x = torch.empty(n, dim, device="cuda")
    for s in range(0, n, CHUNK):
        e = min(n, s + CHUNK)
        if case["kind"] == "graph":  # clusters of neighbouring rows; _links shuffles them
            label = torch.arange(s, e, device="cuda") // TOPIC
        else:
            label = torch.randint(0, clusters, (e - s,), generator=g, device="cuda")
        block = torch.randn(e - s, dim, generator=g, device="cuda").mul_(sigma).add_(centres[label])
        if metric != "l2":
            block /= block.norm(dim=1, keepdim=True)
        if metric == "dot":
            block *= torch.rand(e - s, 1, generator=g, device="cuda") + 0.5
        x[s:e] = block
    pick = torch.randint(0, n, (nq,), generator=g, device="cuda")
    q = x[pick] + noise * torch.randn(nq, dim, generator=g, device="cuda")
    if metric == "cosine":
        q /= q.norm(dim=1, keepdim=True)
    return x, q.contiguous(), g


def _links(x, case, g):
    """A layer-0 adjacency: half of a row's links are its nearest rows (found
    inside its cluster), half lead anywhere; the rows come in random order."""
    n, degree = case["n"], case["degree"]
    near, size = degree // 2, TOPIC
    blocks = n // size
    links = torch.randint(0, n, (n, degree), generator=g, device="cuda")
    for b in range(0, blocks, 256):
        e = min(blocks, b + 256)
        part = x[b * size:e * size].view(e - b, size, -1)
        sim = torch.bmm(part, part.transpose(1, 2).contiguous())
        sim.diagonal(dim1=1, dim2=2).fill_(-2.0)
        best = sim.topk(near, dim=2).indices + (torch.arange(b, e, device="cuda") * size).view(-1, 1, 1)
        links[b * size:e * size, :near] = best.view(-1, near)
    order = torch.randperm(n, generator=g, device="cuda")
    place = torch.empty_like(order)
    place[order] = torch.arange(n, device="cuda")
    return x[order], place[links[order]]


def _new_index(case):
    dim, bits, kind = case["dim"], case.get("bits", 0), case["kind"]
    if kind in ("flat", "rows"):
        return FlatIndex(_context(), dim, case["metric"])
    if kind == "quant":
        return QuantIndex(_context(), dim, bits=bits, scorer=case["scorer"])
    ivf = {"nlist": case["nlist"], "nprobe": case.get("nprobe"), "iters": case.get("iters")}
    return IVFQuantIndex(_context(), dim, bits=bits, ivf=ivf) if bits else IVFIndex(_context(), dim, ivf=ivf)


def prepare(case, seed):
    kind = case["kind"]
    x, q, g = _data(case, seed, case.get("nq", 1))
    state = dict(case=case)
    if kind == "build":
        torch.cuda.synchronize()
        return dict(state, x=x)
    if kind == "graph":
        x, links = _links(x, case, g)
        searcher = GraphSearcher(_context(), case["dim"], "cosine", case["degree"])
        searcher.append(x.cpu().numpy(), case["n"])
        searcher.upload_graph(links.cpu().numpy().astype(np.uint32), case["n"])
        return dict(state, graph=searcher, q=q.cpu().numpy())
    if kind == "rows":
        state["list"] = torch.randperm(case["n"], generator=g, device="cuda")[:case["n_list"]].sort().values.cpu() \
            .numpy().astype(np.uint32)
    index = _new_index(case)
    torch.cuda.synchronize()
    index.append_device(x.data_ptr(), case["n"])
    if kind == "ivf":
        index.build()
    index.sync()
    state["index"] = index
    if kind == "rows" or case["host"]:
        return dict(state, q=q.cpu().numpy())
    nq, k = case["nq"], case["k"]
    return dict(state, q=q, rows=torch.empty(nq, k, dtype=torch.int32, device="cuda"),
                scores=torch.empty(nq, k, dtype=torch.float32, device="cuda"),
                n=torch.empty(nq, dtype=torch.int32, device="cuda"))


# --------------------------------------------------------------------- run --
def run(state):
    case = state["case"]
    kind, k = case["kind"], case.get("k")
    if kind == "build":
        index = _new_index(case)
        index.append_device(state["x"].data_ptr(), case["n"])
        index.build()
        centroids, offsets, rows = index.export_ivf()
        index.destroy()
        return dict(centroids=centroids, offsets=offsets, rows=rows)
    if kind == "graph":
        rows, scores, n = state["graph"].search_arrays(state["q"], case["nq"], k, case["ef"], 0)
        return dict(rows=rows, scores=scores, n=n)
    index, q = state["index"], state["q"]
    if kind == "rows":
        hits = index.query_rows(q, state["list"], k)
        return dict(rows=np.array([h.row for h in hits], np.int64), scores=np.array([h.score for h in hits], np.float32))
    fetch = case.get("fetch", 0)
    if case["host"]:
        rows, scores, n = index.search(q, fetch, k)
        return dict(rows=rows, scores=scores, n=n)
    index.search_device(q.data_ptr(), case["nq"], fetch, k, state["rows"].data_ptr(), state["scores"].data_ptr(),
                        state["n"].data_ptr())
    return dict(rows=state["rows"], scores=state["scores"], n=state["n"])


# -------------------------------------------------------------------- work --
def _padded(dim):
    return 1 << max(2, (dim - 1).bit_length())


def work(case):
    kind, n, dim, bits = case["kind"], case["n"], case["dim"], case.get("bits", 0)
    width = _padded(dim) if bits else dim
    row = width * bits // 8 + 4 if bits else dim * 4  # codes and scale, or the fp32 row
    nq, k, fetch = case.get("nq", 1), case.get("k", 0), case.get("fetch", 0)
    ends = nq * (dim * 4 + k * 8 + 4) + nq * fetch * dim * 4  # queries in, results out, the re-rank's rows
    if kind in ("flat", "quant"):
        return dict(bytes=n * row + ends, flops=2 * nq * n * width + 2 * nq * fetch * dim)
    if kind == "ivf":
        nlist, nprobe = case["nlist"], case["nprobe"]
        probed = n * (1 - (1 - nprobe / nlist) ** nq)  # rows of the lists that any query probes
        return dict(bytes=nlist * width * 4 + probed * (row + 4) + ends,
                    flops=2 * nq * (nlist * width + nprobe / nlist * n * width + fetch * dim))
    if kind == "rows":
        return dict(bytes=case["n_list"] * (dim * 4 + 4) + ends, flops=2 * case["n_list"] * dim)
    if kind == "build":
        train, nlist = min(n, 16384), case["nlist"]
        return dict(bytes=2 * n * dim * 4 + (n * row if bits else 0) + nlist * width * 4 + n * 4,
                    flops=2 * nlist * width * (case["iters"] * train + n))
    # graph: each of the ef expansions reads its links, and about half of them
    # are rows not seen before, whose distances it needs
    walk = nq * case["ef"] * case["degree"]
    return dict(bytes=walk * 4 + walk // 2 * dim * 4 + ends, flops=2 * (walk // 2) * dim)


# -------------------------------------------------------------- comparison --
def tolerance(case):
    if case["kind"] in ("build", "graph"):
        return "exact"  # the arithmetic and its order are part of the interface: f32 in element order
    if case["kind"] == "flat" or (case["kind"] == "ivf" and not case["bits"]):
        # f32 dot products: sums in another order are a few 1e-7 off, and rows
        # closer than that may change places
        return dict(rel=2e-6, max=2e-4, differ=0.004)
    # f64 sums rounded to f32
    return dict(rel=4e-7, max=1e-5, differ=0.0)


def _signs(width, rounds=2):
    """The rotation's signs: one mulberry32 stream per round."""
    out = []
    for r in range(rounds):
        a = SEED ^ (SEED * (r + 1) & 0xFFFFFFFF)
        row = []
        for _ in range(width):
            a = (a + 0x6D2B79F5) & 0xFFFFFFFF
            t = (a ^ (a >> 15)) * (a | 1) & 0xFFFFFFFF
            t ^= (t + ((t ^ (t >> 7)) * (t | 61) & 0xFFFFFFFF)) & 0xFFFFFFFF
            row.append(-1.0 if (t ^ (t >> 14)) < 0x80000000 else 1.0)
        out.append(row)
    return torch.tensor(out, dtype=torch.float64, device="cuda")


def _rotate(x, width, signs):
    """Zero-pad to `width`, then per round signs and an orthonormal Hadamard product."""
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while h.shape[0] < width:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    h = h / math.sqrt(width)
    x = torch.nn.functional.pad(x.double(), (0, width - x.shape[1]))
    for s in signs:
        x = (x * s) @ h
    return x


def _best(keys, first, best, k):
    """The k best of `best` (keys, rows) and of these keys, whose rows begin at `first`."""
    v, i = keys.topk(min(k, keys.shape[1]), dim=1)
    i = i + first
    if best is not None:
        v, i = torch.cat([best[0], v], 1), torch.cat([best[1], i], 1)
        v, at = v.topk(min(k, v.shape[1]), dim=1)
        i = i.gather(1, at)
    return v, i


def exact(case, seed):
    kind, n, dim, k = case["kind"], case["n"], case["dim"], case.get("k")
    if kind not in ("flat", "quant", "rows"):
        return None  # k-means and the graph's walk turn on f32 comparisons; 64 bits would take other turns
    x, q, g = _data(case, seed, case.get("nq", 1))
    qd = q.double()

    def scores(rows):
        rows = rows.double()
        if case.get("metric") == "l2":
            return -(qd.square().sum(1, keepdim=True) + rows.square().sum(1) - 2 * qd @ rows.T)
        return qd @ rows.T

    if kind == "rows":
        at = torch.randperm(n, generator=g, device="cuda")[:case["n_list"]].sort().values
        return dict(rows=None, scores=scores(x[at])[0].topk(min(k, case["n_list"])).values)
    best = None
    if kind == "flat":
        for s in range(0, n, CHUNK):
            best = _best(scores(x[s:s + CHUNK]), s, best, k)
        return dict(rows=None, scores=best[0], n=None)
    bits, width = case["bits"], _padded(dim)
    signs = _signs(width)
    qr = _rotate(q, width, signs)
    if case["scorer"] == "hamming":
        qr = torch.where(qr >= 0, 1.0, -1.0).double()
    for s in range(0, n, CHUNK):
        r = _rotate(x[s:s + CHUNK], width, signs)
        if bits == 1:
            codes, scale = torch.where(r >= 0, 1.0, -1.0).double(), r.abs().mean(1)
        else:
            levels = 127.0 if bits == 8 else 7.0
            scale = r.abs().amax(1)
            codes = torch.floor(r / scale.unsqueeze(1) * levels + 0.5)
        keys = qr @ codes.T
        if case["scorer"] == "hamming":  # whole numbers: ties go to the lower row
            keys -= torch.arange(s, s + keys.shape[1], device="cuda") * 1e-8
        else:
            keys *= scale
        best = _best(keys, s, best, case["fetch"])
    out = torch.stack([(x[rows].double() @ qd[i]).topk(k).values for i, rows in enumerate(best[1])])
    return dict(rows=None, scores=out, n=None)
