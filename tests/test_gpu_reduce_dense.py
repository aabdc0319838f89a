"""The dense reduce of the min-combines on layouts of more than a million
proxies, where it runs from the compute side: no cross mirrors at all, up to
three (loaded together) and up to seven per vertex, several compute partitions,
ragged last words; labels, distances and iteration counts equal the oracle's, by
pulls, by pushes and by both in turn."""
import numpy as np
import pytest

import oracle_lib as O
from grudon_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,deg,C,M", [(1100003, 2.0, 1, 1), (420001, 10.0, 1, 4), (300007, 12.0, 1, 8),
                                       (250003, 12.0, 2, 7)])
def test_dense_reduce(ctx, n, deg, C, M):
    print("dense reduce", n, deg, C, M, flush=True)
    g = O.er(n, deg, seed=M).with_weights(5)
    P = O.Partition(g, C, M)
    G = api.Graph.from_csr(ctx, g.rp, g.col, g.w, C=C, M=M)
    assert G.proxies > 1 << 20
    src = int(np.argmax(g.out_degree() > 0))
    for algo, kw, (ref, st) in ((api.CC, {}, P.cc(nthreads=8)), (api.SSSP, {"source": src}, P.sssp(src, nthreads=8)),
                                (api.SSSP, {"source": src, "weighted": True}, P.sssp(src, weighted=True, nthreads=8))):
        S = api.State(G, algo)
        for option in (api.OPT_PULL_DENSE, api.OPT_PUSH_DENSE):
            S.init(sched=api.SCHED_FIXED, fixed_option=option, **kw)
            stats = S.run()
            assert np.array_equal(S.result(), ref), (algo, option)
            assert stats["iterations"] == int(st[0])
        S.init(sched=api.SCHED_HEURISTIC, **kw)
        k = 0
        while S.step(api.OPT_PULL_DENSE if k % 2 else api.OPT_PUSH_SPARSE):
            k += 1
        assert np.array_equal(S.result(), ref), algo
        S.free()
    G.free()
