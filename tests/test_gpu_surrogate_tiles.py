"""Surrogate products at the edges of their 64 x 64 tiles: batches of one row, of
one tile and a row more or less, split batches, and widths that leave padding.

Oracle and kernels round to bfloat16 at the same points and differ by the order
of fp32 sums, which flips a rounding now and then: one flip is 2^-8 of the
rounded value, so a small tensor's gradient may differ by a few 2^-8 = 4e-3.
Targets lie about 3 from the outputs, so the loss differs by less than twice the
outputs' own error over 3 (2e-3).
"""
import numpy as np
import pytest

import mlp_oracle as M
from sedcol import surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,batch", [((1, 64, 1, 1), 1), ((33, 64, 2, 65), 63), ((64, 192, 1, 64), 64),
                                         ((12, 512, 3, 330), 65), ((31, 128, 2, 63), 129), ((32, 64, 1, 130), 577)])
def test_loss_and_gradient_at_tile_edges(gpu_ready, shape, batch):
    rng = np.random.default_rng(batch)
    layers = M.unflatten(surrogate.init_params(rng, shape).astype(np.float64), *shape)
    p = M.flatten([(W, 0.1 * rng.standard_normal(b.size)) for W, b in layers]).astype(np.float32)
    X = rng.standard_normal((batch, shape[0])).astype(np.float32)
    Y = (3.0 + rng.standard_normal((batch, shape[-1]))).astype(np.float32)
    with surrogate.Network(shape, max_batch=640) as n:
        n.set_params(p)
        lg, gg = n.loss_grad(X, Y)
        n.set_data(X, Y)
        lt = n.train(np.tile(np.arange(batch, dtype=np.int32), 2), batch)
    lo, go, _ = M.loss_grad(p.astype(np.float64), X.astype(np.float64), Y.astype(np.float64), shape)
    assert abs(lg - lo) <= 2e-3 * lo
    off = 0
    for Wo, bo in M.unflatten(go, *shape):
        for ref in (Wo.ravel(), bo):
            got = gg[off:off + ref.size].astype(np.float64)
            off += ref.size
            assert np.linalg.norm(got - ref) <= 2e-2 * np.linalg.norm(ref)
    # a training step makes the same forward pass; the next one starts from the updated weights
    assert lt[0] == np.float32(lg) and 0.0 < lt[1] < lt[0]
