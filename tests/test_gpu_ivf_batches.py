"""GPU tests of the list-major IVF scan at the edges of its chunks: rows of one
to four 256-byte chunks and of less, lists longer than the ids staged at a time
and of a few rows, one and two groups of queries per list."""
import numpy as np
import pytest

from oracle import oracle as o
from tests.helpers import clustered, gaussian, need_gpu, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    need_gpu()
    from browservec_amd import DeviceContext

    c = DeviceContext(0)
    yield c
    c.destroy()


@pytest.mark.parametrize("dim,n,nq,nlist,nprobe", [
    (20, 9000, 17, 2, 2), (40, 5000, 8, 64, 3), (100, 4111, 70, 300, 20),
    (200, 6000, 9, 3, 3), (300, 5003, 40, 16, 4), (1000, 5000, 33, 4, 2),
])
@pytest.mark.parametrize("bits", [8, 4])
def test_list_major_equals_singles(ctx, bits, dim, n, nq, nlist, nprobe):
    from browservec_amd import IVFQuantIndex

    say("ivf list-major edges", bits, dim, n, nq, nlist)
    data = clustered(n, dim, 20, 0.3, seed=dim + nq)
    idx = IVFQuantIndex(ctx, dim, bits=bits, ivf={"nlist": nlist, "iters": 2, "nprobe": nprobe})
    idx.append(data, n)
    qs = data[np.arange(nq) * (n // nq)] + gaussian(nq, dim, 11, normalize=False) * 0.05
    qs = np.stack([o.normalize(q) for q in qs]).astype(np.float32)
    for fetch, k in ((40, 10), (0, 25)):
        rows, scores, cnt = idx.search(qs, fetch, k)
        for i in range(nq):
            r1, s1, c1 = idx.search(qs[i:i + 1], fetch, k)
            assert cnt[i] == c1[0], i
            assert np.array_equal(rows[i, :cnt[i]], r1[0, :c1[0]]), i
            assert np.array_equal(scores[i, :cnt[i]].view(np.uint32), s1[0, :c1[0]].view(np.uint32)), i
    idx.destroy()
