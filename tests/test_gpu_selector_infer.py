"""The selector's inference kernel at the edges of its tiles (16 samples), of
the pinned form (4096 samples) and of its grid (16384 samples in flight on 256
CUs) against the FP64 restatement with the same BF16 weights.  Bar: every logit
is a chain of at most 16 + 64 + 64 + 3 FP32 roundings of terms no larger than
the sum of their magnitudes, carried through the layers: 2^-24 * 160 of that sum."""
import numpy as np
import pytest

import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 255, 4080, 4095, 4096, 4097, 16384, 16401])
def test_inference_sizes(ctx, n):
    print("selector inference sizes", n, flush=True)
    rng = np.random.default_rng(n)
    w = M.init(4).astype(np.float32)
    w += rng.normal(scale=0.05, size=w.size).astype(np.float32)
    bits = (w.view(np.uint32) >> 16).astype(np.uint16)
    wf = (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    x = rng.normal(size=(n, 16)).astype(np.float32)
    ctx.selector_load(bits, 0.0)
    got = ctx.selector_infer(x)
    ref, (_, h1, _, h2) = M.forward(wf, x.astype(np.float64))
    p = M.unpack(wf)
    mag = np.abs(x).astype(np.float64) @ np.abs(p["W1"]).T + np.abs(p["b1"])
    mag = mag @ np.abs(p["W2"]).T + np.abs(p["b2"])
    mag = mag @ np.abs(p["W3"]).T + np.abs(p["b3"])
    assert (np.abs(got - ref) <= 160 * 2.0 ** -24 * mag).all()
    assert np.array_equal(ctx.selector_infer(x).view(np.uint32), got.view(np.uint32))
    # a sample's logits do not depend on its place
    k = min(n, 37)
    assert np.array_equal(ctx.selector_infer(x[n - k:]).view(np.uint32), got[n - k:].view(np.uint32))
