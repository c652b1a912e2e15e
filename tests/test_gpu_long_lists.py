"""GPU tests of the batch selection over lists longer than the registers hold:
IVF batches whose candidates number a few above 16,384, many times that, and
many equal scores, against the same queries run one at a time."""
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


@pytest.mark.parametrize("n,dup,fetch,k", [(16_390, 1, 40, 10), (70_000, 1, 1024, 10), (70_000, 1, 1, 1),
                                           (60_000, 20_000, 100, 10), (40_000, 500, 1000, 100)])
@pytest.mark.parametrize("bits", [8, 4])
def test_long_lists(ctx, bits, n, dup, fetch, k):
    """dup: copies of each row (equal scores go to the lower row)."""
    from browservec_amd import IVFQuantIndex

    say("selection over long lists", bits, n, dup, fetch, k)
    dim, nq = 64, 9
    data = np.tile(clustered(max(n // dup, 1), dim, 8, 0.4, seed=n + dup), (dup, 1))[:n]
    idx = IVFQuantIndex(ctx, dim, bits=bits, ivf={"nlist": 2, "iters": 2, "nprobe": 2})
    idx.append(data, len(data))
    qs = np.stack([o.normalize(q) for q in gaussian(nq, dim, 5)]).astype(np.float32)
    rows, scores, cnt = idx.search(qs, fetch, k)
    for i in range(nq):
        r1, s1, c1 = idx.search(qs[i:i + 1], fetch, k)
        assert cnt[i] == c1[0] == min(k, fetch), i
        assert np.array_equal(rows[i, :cnt[i]], r1[0, :c1[0]]), i
        assert np.array_equal(scores[i, :cnt[i]].view(np.uint32), s1[0, :c1[0]].view(np.uint32)), i
    idx.destroy()
