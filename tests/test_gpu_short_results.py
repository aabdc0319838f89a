"""Results at the edges of the short download (16384 values in parts of 4096, and
65536 through the small pinned buffer):
4- and 8-byte labels and distances bit for bit, ranks within their bound, on
graphs with isolated vertices, in one and in several partitions."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 64, 4095, 4096, 4097, 16383, 16384, 16385, 65535, 65536, 65537])
@pytest.mark.parametrize("C,M", [(1, 1), (2, 3)])
def test_short_results(ctx, n, C, M):
    print("short results", n, C, M, flush=True)
    rng = np.random.default_rng(n)
    a, b = rng.integers(0, n, 2 * n), rng.integers(0, n, 2 * n)
    edges = sorted({(int(x), int(y)) for x, y in zip(a, b) if x != y and x % 5 and y % 5})
    g = O.from_edges(n, edges)
    P = O.Partition(g, C, M)
    G = api.Graph.from_csr(ctx, g.rp, g.col, C=C, M=M)
    for vb in (4, 8):
        for algo, kw, ref in ((api.CC, {}, P.cc()[0]), (api.SSSP, {"source": n // 2}, P.sssp(n // 2)[0])):
            S = api.State(G, algo, vb)
            S.init(sched=api.SCHED_HEURISTIC, **kw)
            S.run()
            want = ref.astype(np.uint64)
            if vb == 8:
                want[ref == 0xFFFFFFFF] = np.uint64(2 ** 64 - 1)
            for _ in range(2):
                assert np.array_equal(S.result().astype(np.uint64), want)
            S.free()
    S = api.State(G, api.PR_PULL)
    S.init(tolerance=1e-6)
    st = S.run()
    ref, _, _ = O.pr_pull(g, iters=st["iterations"])
    assert np.abs(S.result().astype(np.float64) - ref).sum() <= 1e-6
    S.free()
    G.free()
