"""The selector's gradient kernel at the edges of its split (four waves to a
block, a block per CU: 1024 samples at once on 256 CUs) against the FP64
restatement, at the bar of the gradient test (1e-4 of the largest entry), and
bit for bit from run to run."""
import numpy as np
import pytest

import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 255, 1023, 1024, 1025, 2049])
def test_gradient_sizes(ctx, n):
    print("selector gradient sizes", n, flush=True)
    rng = np.random.default_rng(n)
    w = M.init(2).astype(np.float32)
    x = rng.normal(size=(n, 16)).astype(np.float32)
    y = rng.integers(0, 4, size=n).astype(np.uint32)
    for sw in (None, rng.uniform(0.2, 3.0, size=n).astype(np.float32)):
        loss, g = ctx.selector_grad(w, x, y, sw)
        loss64, g64 = M.loss_grad(w.astype(np.float64), x, y.astype(np.int64), sw)
        assert abs(loss - loss64) <= 1e-4 * abs(loss64)
        assert np.abs(g - g64).max() <= 1e-4 * np.abs(g64).max()
        loss2, g2 = ctx.selector_grad(w, x, y, sw)
        assert loss2 == loss and np.array_equal(g2.view(np.uint32), g.view(np.uint32))
