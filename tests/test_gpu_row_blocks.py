"""The row-block pull against the oracle, as the default pull of a small graph
and by mode 0: rows at the edges of the lane groups, of the wave-wide sums and
marks (64 arcs a lane) and of a block (2048 arcs), among rows of a few arcs, so
that long rows share a block with many short ones; and the line up to which the
default takes it."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api
from test_gpu_cold import _graph

pytestmark = pytest.mark.gpu

ROWS = [0, 1, 2, 63, 64, 65, 66, 127, 128, 129, 130, 255, 1000, 1500, 1, 0, 1900, 2047, 2048, 2049, 4100]


@pytest.mark.parametrize("mode", [0, 3])
@pytest.mark.parametrize("C,M", [(1, 1), (1, 4), (2, 3)])
@pytest.mark.parametrize("n,extra", [(5003, 1), (5003, 12), (40009, 3)])
def test_row_block_pull(ctx, mode, C, M, n, extra):
    print("row-block pull", mode, C, M, n, extra, flush=True)
    gw = _graph(n, ROWS, extra, n + extra).with_weights(7)
    P = O.Partition(gw, C, M)
    ctx.set_pull_tiling(mode, 0, 0)
    try:
        G = api.Graph.from_csr(ctx, gw.rp, gw.col, gw.w, C=C, M=M)
        for algo, kw, (ref, st) in ((api.CC, {}, P.cc(nthreads=4)), (api.SSSP, {"source": 3}, P.sssp(3, nthreads=4)),
                                    (api.SSSP, {"source": 3, "weighted": True}, P.sssp(3, weighted=True, nthreads=4))):
            for every in (False, True):
                for option in (api.OPT_PULL_SPARSE, api.OPT_PULL_DENSE):
                    S = api.State(G, algo)
                    S.init(sched=api.SCHED_FIXED, fixed_option=option, pull_every_row=every, **kw)
                    stats = S.run()
                    assert np.array_equal(S.result(), ref)
                    assert stats["iterations"] == int(st[0])
                    S.free()
        S = api.State(G, api.PR)
        S.init(sched=api.SCHED_FIXED, fixed_option=api.OPT_PULL_DENSE)
        S.run()
        out = S.result().astype(np.float64)
        ref64, _ = P.pr(fp64=True, nthreads=4)
        ref32, _ = P.pr(fp64=False, nthreads=4)
        l1 = np.abs(out / out.sum() - ref64 / ref64.sum()).sum()
        l1_32 = np.abs(ref32 / ref32.sum() - ref64 / ref64.sum()).sum()
        assert l1 <= max(1e-6, 4 * l1_32)  # the bound of the reference-PageRank parity test
        S.free()
        S = api.State(G, api.PR_PULL)
        S.init(tolerance=1e-6)
        stats = S.run()
        ref, _, _ = O.pr_pull(gw, iters=stats["iterations"], nthreads=4)
        assert np.abs(S.result().astype(np.float64) - ref).sum() <= 1e-6
        S.free()
        assert G.info()[11:15] == [0, 0, 0, 0]  # nothing was regrouped
        G.free()
    finally:
        ctx.set_pull_tiling(3, 0, 0)


def test_default_pull_by_size(ctx):
    """A graph just beyond the sums' line is split for PageRank and not for CC;
    an explicit window splits the smallest."""
    print("default pull by size", flush=True)
    g = O.rmat(18, 32, seed=5)
    assert 6 << 20 < int(g.rp[-1]) < 16 << 20
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=1)
    S = api.State(G, api.CC)
    assert G.info()[11:15] == [0, 0, 0, 0]
    S.free()
    S = api.State(G, api.PR)
    assert G.info()[11:15] != [0, 0, 0, 0]
    S.free()
    ref, st = O.Partition(g, 1, 1).cc(nthreads=4)
    S = api.State(G, api.CC)  # (the split is there; the line still holds)
    S.init(sched=api.SCHED_FIXED, fixed_option=api.OPT_PULL_DENSE)
    S.run()
    assert np.array_equal(S.result(), ref)
    S.free()
    G.free()
    g = O.rmat(10, 8, seed=5)
    ctx.set_pull_tiling(3, 15, 0)
    try:
        G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=1)
        S = api.State(G, api.CC)
        assert G.info()[11:15] != [0, 0, 0, 0]
        S.free()
        G.free()
    finally:
        ctx.set_pull_tiling(3, 0, 0)
