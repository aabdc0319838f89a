"""The superstep's entry points called more than once, or later than usual,
after one broadcast (the operator API's gen_updates is such a call): results
against the oracle on graphs of which every vertex has enough out-arcs for the
push's heavy list."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu

DEGREES = [64, 20, 65, 257, 64]


def _graph(n):
    """Vertex v points at the DEGREES[v % 5] vertices after it, 7 apart."""
    deg = np.array(DEGREES)[np.arange(n) % len(DEGREES)]
    src = np.repeat(np.arange(n), deg)
    k = np.arange(len(src)) - np.repeat(np.cumsum(deg) - deg, deg)
    keys = np.unique(src.astype(np.int64) * n + (src + 1 + 7 * k) % n)
    rp = np.concatenate([[0], np.cumsum(np.bincount(keys // n, minlength=n))])
    return O.Graph(rp.astype(np.uint32), (keys % n).astype(np.uint32))


def _call(name, S, *args):
    api._check(getattr(api.lib(), name)(S.h, *args), name)


@pytest.mark.parametrize("M", [1, 3])
@pytest.mark.parametrize("option", [api.OPT_PUSH_SPARSE, api.OPT_PUSH_DENSE, api.OPT_SHIP_EDGES])
def test_push_traversal_repeated(ctx, M, option):
    """Two and three traversals of one broadcast: the min-combine's labels are
    those of one, the sums count every arc as often as it was traversed."""
    print("push traversal repeated", M, option, flush=True)
    g = _graph(3001)
    ref, st = O.Partition(g, 1, M).cc()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=M)
    S = api.State(G, api.CC)
    S.init()
    steps, left = 0, 1
    while left:
        _call("grd_broadcast", S, option)
        for _ in range(3):
            _call("grd_traverse", S, option)
        _call("grd_reduce", S, option)
        left = S.step_update()
        steps += 1
    assert np.array_equal(S.result(), ref) and steps == int(st[0])
    S.free()
    S = api.State(G, api.PR)
    S.init()
    _call("grd_broadcast", S, option)
    for _ in range(2):
        _call("grd_traverse", S, option)
    _call("grd_reduce", S, option)
    S.step_update()
    deg = np.diff(g.rp.astype(np.int64))
    src = np.repeat(np.arange(g.n), deg)
    upd = 2 * np.bincount(g.col, weights=0.85 * 0.15 / deg[src], minlength=g.n)
    want = 0.15 + upd
    terms = 2 * np.bincount(g.col, minlength=g.n)
    # FP32 addends of two roundings each, summed in any order, and the last sum
    assert (np.abs(S.result() - want) <= (terms + 4) * 2.0 ** -24 * want).all()
    S.free()
    G.free()


def test_reduce_after_the_update(ctx):
    """A reduce that follows its superstep's update belongs to no superstep of
    the run after it: the run's first one (an empty frontier) has sent nothing,
    and the run ends with the oracle's labels."""
    print("reduce after the update", flush=True)
    g = O.rmat(10, 8, seed=5, symmetrize=True)
    ref, _ = O.Partition(g, 1, 2).cc()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=2)
    S = api.State(G, api.CC)
    S.init(sched=api.SCHED_FIXED, fixed_option=api.OPT_PUSH_SPARSE)
    _call("grd_broadcast", S, api.OPT_PUSH_SPARSE)
    _call("grd_traverse", S, api.OPT_PUSH_SPARSE)
    assert S.step_update() == 0  # nothing has been reduced
    _call("grd_reduce", S, api.OPT_PUSH_SPARSE)
    _, trace = S.run(trace_cap=50)
    assert trace[1].frontier == 0 and trace[1].dirty == 0
    assert np.array_equal(S.result(), ref)
    S.free()
    G.free()


@pytest.mark.parametrize("M", [1, 3])
@pytest.mark.parametrize("option", [api.OPT_PUSH_SPARSE, api.OPT_PUSH_DENSE])
def test_push_traversal_after_the_update(ctx, M, option):
    """A push traversal pushes the frontier that was broadcast, heavy vertices
    included, also when an update has come between (and found nothing)."""
    print("push traversal after the update", M, option, flush=True)
    g = _graph(3001)
    ref, st = O.Partition(g, 1, M).cc()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=M)
    S = api.State(G, api.CC)
    S.init(sched=api.SCHED_FIXED, fixed_option=option)
    _call("grd_broadcast", S, option)
    assert S.step_update() == 0
    _call("grd_traverse", S, option)
    _call("grd_reduce", S, option)
    S.step_update()
    stats = S.run()
    assert np.array_equal(S.result(), ref)
    assert stats["iterations"] == int(st[0]) + 1 and stats["edges_examined"] == int(st[2])
    S.free()
    G.free()


@pytest.mark.parametrize("mode,tb", [(0, 0), (3, 4), (3, 8)])
@pytest.mark.parametrize("option", [api.OPT_PULL_SPARSE, api.OPT_PULL_DENSE])
@pytest.mark.parametrize("algo", ["cc", "hop", "weighted"])
def test_pull_traversal_after_the_update(ctx, mode, tb, option, algo):
    """A pull traversal pulls what was broadcast also when an update has come
    between (and found nothing): in the first superstep and in the second,
    which leaves out rows that cannot improve."""
    print("pull traversal after the update", mode, tb, option, algo, flush=True)
    g = O.rmat(12, 16, seed=5, symmetrize=True).with_weights(11)
    P = O.Partition(g, 1, 2)
    kw = {"cc": {}, "hop": {"source": 3}, "weighted": {"source": 3, "weighted": True}}[algo]
    ref, st = P.cc() if algo == "cc" else P.sssp(3, weighted=algo == "weighted")
    ctx.set_pull_tiling(mode, tb, 0)
    try:
        G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=1, M=2)
        for before in (0, 1):
            S = api.State(G, api.CC if algo == "cc" else api.SSSP)
            S.init(sched=api.SCHED_FIXED, fixed_option=option, **kw)
            for _ in range(before):
                S.step(option)
            _call("grd_broadcast", S, option)
            assert S.step_update() == 0
            _call("grd_traverse", S, option)
            _call("grd_reduce", S, option)
            S.step_update()
            stats = S.run()
            assert np.array_equal(S.result(), ref)
            assert stats["iterations"] == int(st[0]) + 1
            S.free()
        G.free()
    finally:
        ctx.set_pull_tiling(3, 0, 0)  # the default


@pytest.mark.parametrize("C", [1, 2])
def test_shipping_a_stale_list_is_refused(ctx, C):
    """Edge shipping after an update, whose frontier is another one than the
    list that was broadcast, is refused, and the state goes on as if it had not
    been called."""
    print("stale shipping", C, flush=True)
    # even and odd vertices apart, so that two compute partitions cover theirs
    v = np.arange(2000)
    g = O.from_edges(2000, [(int(a), int(b)) for a in v for b in ((a + 2) % 2000, a // 4 * 2 + a % 2) if a != b])
    ref, st = O.Partition(g, C, 2).cc()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=C, M=2)
    assert G.coverage()[1] == 0
    S = api.State(G, api.CC)
    S.init(sched=api.SCHED_FIXED, fixed_option=api.OPT_SHIP_EDGES)
    left = S.step(api.OPT_SHIP_EDGES)
    assert 0 < left < 2000
    with pytest.raises(api.GrdError):
        _call("grd_traverse", S, api.OPT_SHIP_EDGES)
        S.step_update()
    stats = S.run()
    assert np.array_equal(S.result(), ref) and stats["iterations"] == int(st[0])
    S.free()
    G.free()


@pytest.mark.parametrize("degree", [8, 70])
def test_shipping_after_the_update_ships_the_present_values(ctx, degree):
    """Edge shipping aggregates what the compute side holds: after an update whose
    frontier is again every vertex, the values of that update and not those that
    were broadcast (light and heavy vertices)."""
    print("shipping after the update", degree, flush=True)
    n = 500
    src = np.repeat(np.arange(n), degree)
    dst = (src + np.tile(np.arange(1, degree + 1), n)) % n
    col = dst.reshape(n, degree)
    col.sort(axis=1)
    G = api.Graph.from_csr(ctx, (np.arange(n + 1) * degree).astype(np.uint32), col.ravel().astype(np.uint32), C=1, M=2)
    S = api.State(G, api.PR)
    S.init()
    assert S.step(api.OPT_SHIP_EDGES) == n
    _call("grd_traverse", S, api.OPT_SHIP_EDGES)
    assert S.step_update() == n
    # every vertex gets its in-neighbours' 0.85 u / degree, `degree` of them
    want = 0.15 * (1 + 0.85 + 0.85 ** 2)
    assert (np.abs(S.result() - want) <= (3 * degree + 8) * 2.0 ** -24 * want).all()
    S.free()
    G.free()
