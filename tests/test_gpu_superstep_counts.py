"""Counts of a superstep taken apart: what a snapshot within a superstep, a
repeated pull traversal and an earlier state on the same context leave in the
statistics (edges, exchanged bytes, features, residual)."""
import ctypes as ct

import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu


def _call(name, S, *args):
    api._check(getattr(api.lib(), name)(S.h, *args), name)


def _stats(S):
    st = api.RunStats()
    _call("grd_state_stats", S, ct.byref(st))
    return st.as_dict()


def _graph():
    return O.rmat(12, 16, seed=5, symmetrize=True)


@pytest.mark.parametrize("option", [api.OPT_PUSH_SPARSE, api.OPT_PULL_SPARSE])
def test_snapshot_between_reduce_and_update(ctx, option):
    """An update after the restore counts what the first one counted: the dirty
    proxies (a feature, and the bytes of a sparse reduce) and the arcs left out."""
    print("snapshot between reduce and update", option, flush=True)
    g = _graph()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=2)
    S = api.State(G, api.CC)
    S.init()
    S.step(option)
    for name in ("grd_broadcast", "grd_traverse", "grd_reduce"):
        _call(name, S, option)
    S.snapshot()
    left = S.step_update()
    want, feat = _stats(S), S.features()
    assert feat[4] > 0  # dirty proxies
    for _ in range(2):
        S.restore()
        assert S.step_update() == left
        got = _stats(S)
        assert [got[k] for k in ("bytes_exchanged", "edges_examined")] == \
               [want[k] for k in ("bytes_exchanged", "edges_examined")]
        assert np.array_equal(S.features(), feat)
    S.free()
    G.free()


@pytest.mark.parametrize("mode,tb", [(0, 0), (3, 4)])
def test_repeated_pull_counts_twice(ctx, mode, tb):
    """Two pull traversals of one broadcast examine twice the arcs of one, less
    twice those that were left out."""
    print("repeated pull", mode, tb, flush=True)
    g = _graph()
    ctx.set_pull_tiling(mode, tb, 0)
    try:
        G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=2)
        S = api.State(G, api.CC)
        edges = []
        for times in (1, 2, 3):
            S.init()
            S.step(api.OPT_PULL_DENSE)
            before = _stats(S)["edges_examined"]
            _call("grd_broadcast", S, api.OPT_PULL_DENSE)
            for _ in range(times):
                _call("grd_traverse", S, api.OPT_PULL_DENSE)
            _call("grd_reduce", S, api.OPT_PULL_DENSE)
            S.step_update()
            edges.append(_stats(S)["edges_examined"] - before)
        assert 0 < edges[0] < g.m  # some arcs were left out
        assert edges[1:] == [2 * edges[0], 3 * edges[0]]
        S.free()
        G.free()
    finally:
        ctx.set_pull_tiling(3, 0, 0)  # the default


def test_residual_is_pull_pageranks(ctx):
    """The residual of another state, whose memory a new one got, is not the new
    one's: an algorithm without a residual reports none."""
    print("residual", flush=True)
    g = _graph()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=2)
    for algo in (api.CC, api.PR, api.SSSP):
        S = api.State(G, api.PR_PULL)
        S.init(max_iter=2)
        S.run()
        assert _stats(S)["residual"] > 0
        S.free()
        S = api.State(G, algo)
        S.init(max_iter=2)
        S.run()
        assert _stats(S)["residual"] == 0
        S.free()
    G.free()


@pytest.mark.parametrize("mode,tb", [(0, 0), (3, 4), (3, 8)])
@pytest.mark.parametrize("algo", ["cc", "weighted"])
def test_pull_after_the_update_marks_nothing(ctx, mode, tb, algo):
    """A pull traversal that repeats the superstep's own after its update leaves
    out the same rows, finds the same values and so marks no proxy for the next
    reduce."""
    print("pull after the update", mode, tb, algo, flush=True)
    g = _graph().with_weights(11)
    ctx.set_pull_tiling(mode, tb, 0)
    try:
        G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=1, M=2)
        seen = []
        for extra in (0, 1, 2):
            S = api.State(G, api.CC if algo == "cc" else api.SSSP)
            S.init(source=3, weighted=algo != "cc")
            steps = []
            for _ in range(3):
                S.step(api.OPT_PULL_SPARSE)
                for _ in range(extra):
                    _call("grd_traverse", S, api.OPT_PULL_SPARSE)
                steps.append((_stats(S)["bytes_exchanged"], S.features().tolist()))
            seen.append(steps)
            S.free()
        assert seen[1] == seen[0] and seen[2] == seen[0]
        G.free()
    finally:
        ctx.set_pull_tiling(3, 0, 0)  # the default
