"""The cold pass of the hot / cold pull against the oracle: rows at the edges of
the wave-wide row sums and of the block sizes (2048, 4096 and 16384 arcs; the
last two on a graph of more than 2^20 vertices in one partition, where they are
used), with a 16-source window so that nearly every arc is cold."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu

SMALL = [0, 1, 2, 23, 24, 25, 47, 48, 49, 63, 64, 65, 255, 2047, 2048, 2049, 4100]
LARGE = [4095, 4096, 4097, 16383, 16384, 16385, 40000]


def _graph(n, rows, extra, seed):
    """Row v < len(rows) has rows[v] in-arcs from distinct sources; the others
    `extra` random in-arcs each on average."""
    rng = np.random.default_rng(seed)
    s, d = [rng.integers(0, n, extra * n)], [rng.integers(0, n, extra * n)]
    keep = d[0] >= len(rows)
    s, d = [s[0][keep]], [d[0][keep]]
    for v, k in enumerate(rows):
        src = rng.choice(n - 1, size=min(k, n - 1), replace=False) + 1
        src = np.where(src == v, 0, src) if v else src
        s.append(src)
        d.append(np.full(len(src), v))
    s, d = np.concatenate(s).astype(np.int64), np.concatenate(d).astype(np.int64)
    keys = np.unique((s * n + d)[s != d])
    rp = np.zeros(n + 1, dtype=np.int64)
    np.add.at(rp, keys // n + 1, 1)
    return O.Graph(np.cumsum(rp).astype(np.uint32), (keys % n).astype(np.uint32))


def _check(ctx, g, M, option):
    gw = g.with_weights(11)
    ctx.set_pull_tiling(3, 4, 0)
    try:
        G = api.Graph.from_csr(ctx, gw.rp, gw.col, gw.w, C=1, M=M)
        P = O.Partition(gw, 1, M)
        for algo, kw, (ref, st) in ((api.CC, {}, P.cc(nthreads=8)), (api.SSSP, {"source": 3}, P.sssp(3, nthreads=8)),
                                    (api.SSSP, {"source": 3, "weighted": True}, P.sssp(3, weighted=True, nthreads=8))):
            for every in (False, True):
                S = api.State(G, algo)
                S.init(sched=api.SCHED_FIXED, fixed_option=option, pull_every_row=every, **kw)
                stats = S.run()
                assert np.array_equal(S.result(), ref)
                assert stats["iterations"] == int(st[0])
                S.free()
        S = api.State(G, api.PR)
        S.init(sched=api.SCHED_FIXED, fixed_option=option)
        S.run()
        out = S.result().astype(np.float64)
        ref64, _ = P.pr(fp64=True, nthreads=8)
        ref32, _ = P.pr(fp64=False, nthreads=8)
        l1 = np.abs(out / out.sum() - ref64 / ref64.sum()).sum()
        l1_32 = np.abs(ref32 / ref32.sum() - ref64 / ref64.sum()).sum()
        assert l1 <= max(1e-6, 4 * l1_32)  # the bound of the reference-PageRank parity test
        S.free()
        S = api.State(G, api.PR_PULL)
        S.init(tolerance=1e-6)
        st = S.run()
        out = S.result()
        ref, _, _ = O.pr_pull(g, iters=st["iterations"], nthreads=8)
        assert np.abs(out.astype(np.float64) - ref).sum() <= 1e-6
        S.init(tolerance=1e-6)
        S.run()
        assert np.array_equal(S.result().view(np.uint32), out.view(np.uint32))  # deterministic
        S.free()
        G.free()
    finally:
        ctx.set_pull_tiling(3, 0, 0)  # the default


@pytest.mark.parametrize("M", [1, 3])
@pytest.mark.parametrize("option", [api.OPT_PULL_SPARSE, api.OPT_PULL_DENSE])
def test_cold_rows_small_blocks(ctx, M, option):
    print("cold rows, blocks of 2048", M, option, flush=True)
    _check(ctx, _graph(6007, SMALL, 3, 2), M, option)


def test_cold_rows_large_blocks(ctx):
    print("cold rows, blocks of 4096 and 16384", flush=True)
    _check(ctx, _graph(1 << 20 | 77, SMALL + LARGE, 2, 3), 1, api.OPT_PULL_DENSE)
