"""GPU test of graph searches that find fewer hits than asked for: the places
past a query's count hold zeros, whatever the arrays and the searcher's buffers
held before."""
import ctypes

import numpy as np
import pytest

from tests.helpers import gaussian, need_gpu, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,ef", [(3, 10, 16), (3, 300, 16), (40, 20, 8)])
def test_places_past_the_count_are_zero(n, k, ef):
    need_gpu()
    from browservec_amd import DeviceContext, GraphSearcher

    say("graph counts", n, k, ef)
    ctx = DeviceContext(0)
    dim, nq = 24, 5
    g = GraphSearcher(ctx, dim, "cosine", 4)
    g.append(gaussian(n, dim, 1), n)
    g.upload_graph(np.array([[(i + j + 1) % n for j in range(4)] for i in range(n)], np.uint32), n)
    qs = np.ascontiguousarray(gaussian(nq, dim, 2), np.float32)
    for _ in range(2):
        rows = np.full((nq, k), 77, np.uint32)
        scores = np.full((nq, k), 7.0, np.float32)
        cnt = np.zeros(nq, np.uint32)
        p = [ctypes.c_void_p(a.ctypes.data) for a in (qs, rows, scores, cnt)]
        assert g.lib.bv_graph_search(g.handle, p[0], nq, k, ef, 0, p[1], p[2], p[3]) == 0
        for i in range(nq):
            assert 0 < cnt[i] <= min(n, k)
            assert not rows[i, cnt[i]:].any() and not scores[i, cnt[i]:].any()
            assert len(set(rows[i, :cnt[i]].tolist())) == cnt[i]
    g.destroy()
    ctx.destroy()
