"""The batched pulls against the oracle at every block size (1024 to 16384 arcs,
chosen from the batch's arcs): rows at the edges of the lane groups, of the
wave-wide row sums and of a block, rows of several blocks, blocks of empty rows,
a graph of one vertex; and the captured iterations under changed parameters."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu

ROWS = [0, 1, 2, 63, 64, 65, 127, 128, 129, 255, 1023, 1024, 1025, 4095, 4096, 4097, 8191, 8192, 8193, 16383, 16384,
        16385, 40000]


def _graph(n, extra, seed):
    """Row v < len(ROWS) has ROWS[v] in-arcs, the next 20000 rows none, the
    others `extra` random ones each."""
    rng = np.random.default_rng(seed)
    first = len(ROWS) + 20000
    s, d = [rng.integers(0, n, extra * n)], [rng.integers(first, n, extra * n)]
    for v, k in enumerate(ROWS):
        s.append(rng.choice(n - len(ROWS), size=k, replace=False) + len(ROWS))
        d.append(np.full(k, v))
    s, d = np.concatenate(s).astype(np.int64), np.concatenate(d).astype(np.int64)
    keys = np.unique((s * n + d)[s != d])
    rp = np.zeros(n + 1, dtype=np.int64)
    np.add.at(rp, keys // n + 1, 1)
    return O.Graph(np.cumsum(rp).astype(np.uint32), (keys % n).astype(np.uint32))


# arcs of the batch: 0.5, 1.4, 2.8, 5.5 and 9.5 M, i.e. blocks of 1024 up to 16384 on 256 CUs
@pytest.mark.parametrize("extra,K", [(3, 1), (11, 4), (23, 3), (46, 8), (82, 2)])
def test_batch_block_sizes(ctx, extra, K):
    print("batch blocks", extra, K, flush=True)
    gs = [_graph(110000, extra, extra), O.from_edges(1, []), O.rmat(10, 8, seed=3)]
    B = api.Batch(ctx, [(g.rp, g.col) for g in gs])
    try:
        B.tune(1024, 8, K)
        first = None
        for damping in (0.85, 0.5, 0.85):
            iters, _ = B.pagerank(damping=damping, tolerance=1e-6, max_iter=200)
            got = [B.result(i, api.PR_PULL) for i in range(B.count)]
            if damping == 0.85:
                for i, g in enumerate(gs):
                    ref, _, _ = O.pr_pull(g, iters=int(iters[i]))
                    assert np.abs(got[i].astype(np.float64) - ref).sum() <= 1e-6, i
                if first is not None:
                    assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(first, got))
                first = got
        iters, _ = B.cc()
        for i, g in enumerate(gs):
            ref, st = O.Partition(g, 1, 1).cc(nthreads=8)
            assert np.array_equal(B.result(i, api.CC), ref), i
            assert int(iters[i]) == int(st[0]), i
    finally:
        B.free()
