"""The hot / cold pull with the default window of 2^15 sources against the
oracle: by an explicit window on graphs whose partitions have more own sources
than the window and on one that lies in it whole, and as the default pull of
graphs above its lines."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu
NT = 8  # oracle threads


@pytest.fixture
def window15(ctx):
    ctx.set_pull_tiling(3, 15, 0)
    yield
    ctx.set_pull_tiling(3, 0, 0)  # the default


def _split(G):
    """(ranges, blocks) of the hot pass: none until a state has split the graph"""
    return G.info()[12] > 0 and G.info()[13] > 0


def _check_pull_pagerank(ctx, G, g):
    S = api.State(G, api.PR_PULL)
    assert _split(G)
    S.init(tolerance=1e-6)
    st = S.run()
    ref, _, _ = O.pr_pull(g, iters=st["iterations"], nthreads=NT)
    assert np.abs(S.result().astype(np.float64) - ref).sum() <= 1e-6
    S.free()


def _check_pagerank(G, P):
    S = api.State(G, api.PR)
    assert _split(G)
    S.init(sched=api.SCHED_FIXED, fixed_option=api.OPT_PULL_DENSE)
    S.run()
    out = S.result().astype(np.float64)
    ref64, _ = P.pr(fp64=True, nthreads=NT)
    ref32, _ = P.pr(fp64=False, nthreads=NT)
    l1 = np.abs(out / out.sum() - ref64 / ref64.sum()).sum()
    l1_32 = np.abs(ref32 / ref32.sum() - ref64 / ref64.sum()).sum()
    assert l1 <= max(1e-6, 4 * l1_32)  # the bound of the reference-PageRank parity test
    S.free()


def _check_mins(G, P, options, weights=(False, True), every=(False, True)):
    for algo, kw, (ref, st) in [(api.CC, {}, P.cc(nthreads=NT))] + \
            [(api.SSSP, {"source": 3, "weighted": w}, P.sssp(3, weighted=w, nthreads=NT)) for w in weights]:
        for option in options:
            for ev in every:
                S = api.State(G, algo)
                assert _split(G)
                S.init(sched=api.SCHED_FIXED, fixed_option=option, pull_every_row=ev, **kw)
                stats = S.run()
                assert np.array_equal(S.result(), ref)
                assert stats["iterations"] == int(st[0])
                S.free()


@pytest.mark.parametrize("scale,C,M", [(10, 1, 2), (16, 1, 4), (17, 1, 1), (18, 2, 3)])
def test_pull_pagerank(ctx, window15, scale, C, M):
    print("window 15, pull PageRank", scale, C, M, flush=True)
    g = O.rmat(scale, 16, seed=scale + 7)
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=C, M=M)
    _check_pull_pagerank(ctx, G, g)
    G.free()


@pytest.mark.parametrize("C,M", [(1, 1), (2, 2)])
@pytest.mark.parametrize("wide", [False, True])
def test_bsp_pull(ctx, window15, C, M, wide):
    """wide: a weight beyond a byte."""
    print("window 15, BSP pull", C, M, wide, flush=True)
    g = O.rmat(17, 16, seed=5, symmetrize=True).with_weights(11)
    if wide:
        g.w[::1000] += 1000
    P = O.Partition(g, C, M)
    G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=C, M=M)
    _check_mins(G, P, (api.OPT_PULL_SPARSE, api.OPT_PULL_DENSE))
    if not wide:
        _check_pagerank(G, P)
    G.free()


def test_flat_degrees(ctx, window15):
    """Every source about as hot as the next: hot rows of a few arcs each."""
    print("window 15, Erdos-Renyi", flush=True)
    g = O.er(100003, 12.0, seed=5)
    P = O.Partition(g, 1, 2)
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=2)
    _check_mins(G, P, (api.OPT_PULL_DENSE,), weights=(False,))
    _check_pull_pagerank(ctx, G, g)
    G.free()


def test_default_beyond_the_sums_line(ctx):
    print("default pull, sums", flush=True)
    g = O.rmat(18, 32, seed=5)
    assert 6 << 20 < g.m < 16 << 20
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=1)
    assert not _split(G)
    _check_pagerank(G, O.Partition(g, 1, 1))
    _check_pull_pagerank(ctx, G, g)
    G.free()


def test_default_beyond_every_line(ctx):
    print("default pull, min-combines", flush=True)
    g = O.rmat(19, 20, seed=5, symmetrize=True).with_weights(11)
    assert g.m > 16 << 20
    G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=1, M=4)
    assert not _split(G)
    _check_mins(G, O.Partition(g, 1, 4), (api.OPT_PULL_DENSE,), weights=(True,), every=(False,))
    G.free()


@pytest.mark.parametrize("bits", [15, 8])
def test_graph_keeps_the_window_asked_for(ctx, bits):
    """States that come after the context is back at its default still pull over
    the graph's own regrouping, as long as that was asked for.  (The split
    stores the weights of this graph as bytes, the row-block pull as words.)"""
    print("window asked for", bits, flush=True)
    g = O.rmat(10, 8, seed=5, symmetrize=True).with_weights(11)

    def weight_bytes(G):
        S = api.State(G, api.SSSP)
        S.init(source=3, weighted=True, sched=api.SCHED_FIXED, fixed_option=api.OPT_PULL_DENSE, max_iter=1,
               time_kernel=True, pull_every_row=True)
        b = S.run()["kernel_bytes"]
        S.free()
        return (b - 8 * G.info()[5]) / g.m - 8

    G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=1, M=2)
    assert weight_bytes(G) == 4  # a small graph's default pull
    ctx.set_pull_tiling(3, bits, 0)
    try:
        assert weight_bytes(G) == 1
    finally:
        ctx.set_pull_tiling(3, 0, 0)  # the default
    assert _split(G) and weight_bytes(G) == 1
    G.free()
