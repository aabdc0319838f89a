"""The push's split of the frontier against the oracle: out-degrees at the
edges of the heavy threshold (64) and of the heavy chunks (256 arcs), tiles
of 64 and of 256 active vertices, ragged last tiles.  CC and SSSP bit-exact
with equal iteration counts."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu

DEGREES = [0, 1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2048, 2049, 5000]


def _hubs(n, seed):
    """Vertex 0 reaches every hub; hub i has DEGREES[i % 14] distinct targets."""
    rng = np.random.default_rng(seed)
    nh = 3 * len(DEGREES)
    edges = [(0, 1 + i) for i in range(nh)]
    for i in range(nh):
        for t in rng.choice(n, size=DEGREES[i % len(DEGREES)], replace=False):
            if t != 1 + i:
                edges.append((1 + i, int(t)))
    edges += [(int(a), int(b)) for a, b in rng.integers(0, n, (4 * n, 2)) if a != b and a > nh]
    return O.from_edges(n, sorted(set(edges)))


@pytest.mark.parametrize("C,M", [(1, 1), (2, 3)])
@pytest.mark.parametrize("option", [api.OPT_PUSH_SPARSE, api.OPT_PUSH_DENSE])
def test_push_degree_edges(ctx, C, M, option):
    print("push degree edges", C, M, option, flush=True)
    g = _hubs(6001, 5).with_weights(7)
    P = O.Partition(g, C, M)
    G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=C, M=M)
    for algo, kw, (ref, st) in ((api.CC, {}, P.cc()), (api.SSSP, {}, P.sssp(0)),
                                (api.SSSP, {"weighted": True}, P.sssp(0, weighted=True))):
        S = api.State(G, algo)
        S.init(sched=api.SCHED_FIXED, fixed_option=option, **kw)
        stats = S.run()
        assert np.array_equal(S.result(), ref)
        assert stats["iterations"] == int(st[0])
        S.free()
    S = api.State(G, api.PR)
    ref64, _ = P.pr(fp64=True)
    ref32, _ = P.pr(fp64=False)
    S.init(sched=api.SCHED_FIXED, fixed_option=option)
    S.run()
    out = S.result().astype(np.float64)
    l1 = np.abs(out / out.sum() - ref64 / ref64.sum()).sum()
    l1_32 = np.abs(ref32 / ref32.sum() - ref64 / ref64.sum()).sum()
    assert l1 <= max(1e-6, 4 * l1_32)  # the bound of the reference-PageRank parity test


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 257, 131071, 131072, 131073, 200003])
def test_push_tile_edges(ctx, n):
    """A frontier of n vertices (CC's first superstep) around the tile sizes
    and around the frontier at which tiles grow from 64 to 256 (131072)."""
    print("push tile edges", n, flush=True)
    v = np.arange(n)
    edges = sorted({(int(a), int(b)) for a, b in zip(v, (v * 7 + 3) % n) if a != b})
    g = O.from_edges(n, edges)
    ref, st = O.Partition(g, 1, 2).cc()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=2)
    S = api.State(G, api.CC)
    S.init(sched=api.SCHED_PLAIN)
    stats = S.run()
    assert np.array_equal(S.result(), ref)
    assert stats["iterations"] == int(st[0])


@pytest.mark.parametrize("n", [524225, 524287, 524288, 524289, 600001])
def test_rank_edges(ctx, n):
    """Bitmaps around 8192 words, where the word ranks turn from one launch to
    three, in sparse pushes and pulls."""
    print("rank edges", n, flush=True)
    v = np.arange(n, dtype=np.uint32)
    rp = np.concatenate([[0], np.maximum(np.arange(1, n + 1) - 1, 0)]).astype(np.uint32)
    g = O.Graph(rp, v[1:] // 2)  # v -> v / 2
    ref, st = O.Partition(g, 1, 2).cc()
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=1, M=2)
    for option in (api.OPT_PUSH_SPARSE, api.OPT_PULL_SPARSE, api.OPT_SHIP_EDGES):
        S = api.State(G, api.CC)
        S.init(sched=api.SCHED_FIXED, fixed_option=option)
        stats = S.run()
        assert np.array_equal(S.result(), ref)
        assert stats["iterations"] == int(st[0])
        S.free()
