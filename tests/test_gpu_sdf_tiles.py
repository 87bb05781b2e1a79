"""The training kernel's gradient at the edges of its 128-sample tiles and of
its blocks (one sample, a tile less and more by one, several tiles per block,
many bodies) against the oracle's binary64 gradient."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bodies,samples", [(1, 1), (1, 127), (2, 128), (1, 129), (3, 1000),
                                            (40, 1025)])
def test_gradient_tiles(gpu_ctx, bodies, samples):
    from fullc0ntact_amd import _lib
    from fullc0ntact_amd.sdf import SdfSurrogate
    print(bodies, samples, flush=True)
    rng = np.random.default_rng(samples)
    s = SdfSurrogate(gpu_ctx, rng.uniform(-0.1, 0.1, (bodies, 3)),
                     rng.uniform(0.8, 1.2, bodies), seed=7)
    p, f, fr = s.params()
    p = p + rng.normal(0.0, 0.03, p.shape).astype(np.float32)
    s.set_params(p)
    pts = rng.uniform(-0.7, 0.7, (bodies, samples, 3)).astype(np.float32)
    lab = rng.uniform(-0.3, 0.3, (bodies, samples)).astype(np.float32)
    dp = _lib.DeviceArray.from_host(gpu_ctx, pts)
    dl = _lib.DeviceArray.from_host(gpu_ctx, lab)
    g, loss = s.loss_grad(dp, dl, samples)
    for b in {0, bodies // 2, bodies - 1}:
        ref, L = orc.sdf_loss_grad(p[b], f[b], fr[b], pts[b], lab[b])
        # binary32 sums of a few hundred terms; the hardware sine and cosine
        assert abs(loss[b] - L) <= 1e-5 * L
        gb = g[b, :s.nparams].astype(np.float64)
        assert np.max(np.abs(gb - ref)) <= 1e-4 * np.max(np.abs(ref))
    s.close()


@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 1000, 32769])
def test_inference_tiles(gpu_ctx, n):
    """Inference at the edges of its 16-query tiles, of its groups of four
    tiles and of one tile per wave; runs of one body, mixed tiles and ids out
    of range."""
    from fullc0ntact_amd.sdf import BF16, SdfSurrogate
    print(n, flush=True)
    rng = np.random.default_rng(n)
    s = SdfSurrogate(gpu_ctx, rng.uniform(-0.1, 0.1, (3, 3)), rng.uniform(0.8, 1.2, 3), seed=7)
    p, f, fr = s.params()
    pts = rng.uniform(-0.8, 0.8, (n, 3)).astype(np.float32)
    bodies = np.where(np.arange(n) < n // 2, 2, rng.integers(0, 4, n)).astype(np.uint32)
    y = s.eval(pts, bodies, BF16)
    assert np.all(np.isnan(y[bodies == 3]))
    for b in range(3):
        m = bodies == b
        if m.any():
            scale = np.max(np.abs(orc.sdf_forward(p[b], f[b], fr[b], pts[:512])))
            ref = orc.sdf_forward(p[b], f[b], fr[b], pts[m], bf16=True)
            # the bound of the whole-network test: BF16 activations that round the other way
            assert np.max(np.abs(y[m] - ref)) <= 2e-3 * max(scale, 0.1), b
    s.close()


@pytest.mark.parametrize("n", [32769, 150001])
def test_inference_is_the_same_in_parts(gpu_ctx, n):
    """A query's distance does not depend on the call it stands in: many tiles
    per wave and mixed tiles against calls of 1,000 queries, bit for bit."""
    from fullc0ntact_amd.sdf import BF16, SdfSurrogate
    print(n, flush=True)
    rng = np.random.default_rng(n)
    s = SdfSurrogate(gpu_ctx, rng.uniform(-0.1, 0.1, (3, 3)), rng.uniform(0.8, 1.2, 3), seed=7)
    pts = rng.uniform(-0.8, 0.8, (n, 3)).astype(np.float32)
    bodies = np.where(np.arange(n) < n // 2, 2, rng.integers(0, 4, n)).astype(np.uint32)
    y = s.eval(pts, bodies, BF16)
    parts = [s.eval(pts[i:i + 1000], bodies[i:i + 1000], BF16) for i in range(0, n, 1000)]
    assert np.array_equal(y.view(np.uint32), np.concatenate(parts).view(np.uint32))
    s.close()


@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 1000, 32769])
def test_fp32_inference_tiles(gpu_ctx, n):
    """The binary32 network at the same edges, mixed tiles and ids out of
    range, and with a query that is not a number beside others."""
    from fullc0ntact_amd.sdf import FP32, SdfSurrogate
    print(n, flush=True)
    rng = np.random.default_rng(n)
    s = SdfSurrogate(gpu_ctx, rng.uniform(-0.1, 0.1, (3, 3)), rng.uniform(0.8, 1.2, 3), seed=7)
    p, f, fr = s.params()
    p = p + rng.normal(0.0, 0.03, p.shape).astype(np.float32)
    s.set_params(p)
    pts = rng.uniform(-0.8, 0.8, (n, 3)).astype(np.float32)
    bodies = np.where(np.arange(n) < n // 2, 2, rng.integers(0, 4, n)).astype(np.uint32)
    lost = (np.arange(n) % 29) == 11
    pts[lost, 1] = np.nan
    y = s.eval(pts, bodies, FP32)
    assert np.array_equal(np.isnan(y), lost | (bodies == 3))
    for b in range(3):
        m = (bodies == b) & ~lost
        if m.any():
            ref = orc.sdf_forward(p[b], f[b], fr[b], pts[m])
            scale = np.max(np.abs(orc.sdf_forward(p[b], f[b], fr[b], pts[~lost][:512])))
            # the bound of the whole-network test: binary32 sums of 64 terms a
            # layer and the hardware sine and cosine (2e-6 of a turn)
            assert np.max(np.abs(y[m] - ref)) <= 1e-4 * max(scale, 0.1), b
    s.close()
