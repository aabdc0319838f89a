"""Pushes whose arcs meet at one vertex (the leaves of a star push to its hub)
against the oracle: whole and partial waves of them, hubs with the smallest and
the largest id, one hub and two among each other's leaves, on the memory side and
shipped."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu


def _star(n, hubs):
    """Every vertex but the hubs is joined with hub v % len(hubs)."""
    h = np.array(hubs)
    v = np.setdiff1d(np.arange(n), h)
    s, d = v, h[v % len(h)]
    keys = np.unique(np.concatenate([s * n + d, d * n + s]))
    rp = np.concatenate([[0], np.cumsum(np.bincount(keys // n, minlength=n))])
    return O.Graph(rp.astype(np.uint32), (keys % n).astype(np.uint32))


@pytest.mark.parametrize("option", [api.OPT_PUSH_SPARSE, api.OPT_PUSH_DENSE, api.OPT_SHIP_EDGES])
@pytest.mark.parametrize("n", [3, 8, 9, 10, 64, 65, 66, 130, 257, 1030, 70001, 300000])
def test_star(ctx, n, option):
    for hubs in ([0], [n - 1], [n // 2, 1]) if n > 4 else ([0], [n - 1]):
        print("star", n, option, hubs, flush=True)
        g = _star(n, hubs).with_weights(5)
        P = O.Partition(g, 1, 2)
        G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=1, M=2)
        src = {"source": 2}
        for algo, kw, (ref, st) in ((api.CC, {}, P.cc(nthreads=4)), (api.SSSP, src, P.sssp(2, nthreads=4)),
                                    (api.SSSP, dict(src, weighted=True), P.sssp(2, weighted=True, nthreads=4))):
            S = api.State(G, algo)
            S.init(sched=api.SCHED_FIXED, fixed_option=option, **kw)
            stats = S.run()
            assert np.array_equal(S.result(), ref)
            assert stats["iterations"] == int(st[0]) and stats["edges_examined"] == int(st[2])
            S.free()
        S = api.State(G, api.PR)
        S.init(sched=api.SCHED_FIXED, fixed_option=option, max_iter=30)
        S.run()
        ref64, _ = P.pr(fp64=True, max_iter=30, nthreads=4)
        ref32, _ = P.pr(fp64=False, max_iter=30, nthreads=4)
        out = S.result().astype(np.float64)
        l1 = np.abs(out / out.sum() - ref64 / ref64.sum()).sum()
        l1_32 = np.abs(ref32 / ref32.sum() - ref64 / ref64.sum()).sum()
        assert l1 <= max(1e-6, 4 * l1_32)  # the bound of the reference-PageRank parity test
        S.free()
        G.free()
