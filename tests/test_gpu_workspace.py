"""Results and inputs through the context's kept buffers: array sizes around
the small buffer (256 KB), the staging slots (4 MB) and their ring, 4- and
8-byte results, and graphs built from blocks that earlier graphs gave back."""
import numpy as np
import pytest

from grudon_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value_bytes", [4, 8])
def test_result_sizes(ctx, value_bytes):
    for n in (1, 63, 65535, 65536, 65537, 1048575, 1048576, 1048577, 5000001):
        print("result size", n, value_bytes, flush=True)
        rp = np.zeros(n + 1, dtype=np.uint32)
        rp[2:] = 1  # one arc, 1 -> 0
        if n < 2:
            rp[:] = 0
        G = api.Graph.from_csr(ctx, rp, np.zeros(int(rp[-1]), dtype=np.uint32), C=1, M=2)
        S = api.State(G, api.CC, value_bytes)
        S.init()
        S.run()
        assert np.array_equal(S.result(), np.arange(n))
        S.free()
        S = api.State(G, api.SSSP, value_bytes)
        S.init(source=n - 1)
        S.run()
        want = np.full(n, (1 << (8 * value_bytes)) - 1, dtype=np.uint64)
        want[n - 1] = 0
        if n == 2:
            want[0] = 1
        assert np.array_equal(S.result().astype(np.uint64), want)
        S.free()
        G.free()


def test_blocks_are_reused_with_other_contents(ctx):
    """The same graphs again after larger and smaller ones, from a context of
    their own: layouts and results must not depend on what a block held."""
    c = api.Context(0)
    try:
        first = {}
        for rnd in range(3):
            for n in (3000, 40000, 700, 40000):
                rp, col = ctx.generate_er(n, 6.0, seed=n)
                G = api.Graph.from_csr(c, rp, col, C=1, M=3)
                S = api.State(G, api.CC)
                S.init(sched=api.SCHED_HEURISTIC)
                S.run()
                got = (G.digest(), S.result())
                S.free()
                G.free()
                want = first.setdefault(n, got)
                print("reuse", rnd, n, flush=True)
                assert np.array_equal(want[0], got[0]) and np.array_equal(want[1], got[1])
    finally:
        c.close()
