"""The training kernels at the batch sizes where their launches are cut differently: one tile, one sample
range and its edges, a second range of one tile, a number of ranges that is no multiple of the eight
XCDs, the largest block.  Gradient and loss against the float64 oracle with the kernels' bf16 rounding
points (float32 accumulation over at most 70,000 terms stays far below the 1e-2 the rounding of single
deltas leaves), every block of parameters, and the loss the same on every call."""
import numpy as np
import pytest

from oracle import guide_oracle as G
from tests.test_guide_gpu import _batch, _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 1000, 1024, 1025, 1088, 9 * 1024 + 65, 20_000, 70_000])
def test_gradient_at_batch_edges(gpu, n):
    g = gpu.Guide(batch_size=70_016)
    th = _params(21)
    g.set_params(th)
    x, d, w = _batch(n, 60 + n)
    w = np.maximum(w, 0.05).astype(np.float32)
    loss, grad = g.grad(x, d, w)
    loss_ref, ref = G.loss_grad(th, x, d, w.astype(np.float64), emulate=True)
    assert np.linalg.norm(grad - ref) / np.linalg.norm(ref) < 1e-2
    for (ow, ob), (rows, cols) in zip(G.OFFSETS, G.SHAPES):
        for lo, hi in ((ow, ob), (ob, ob + rows)):
            assert np.linalg.norm(grad[lo:hi] - ref[lo:hi]) < 3e-2 * max(np.linalg.norm(ref[lo:hi]), 1e-30), (lo, hi)
    assert abs(loss - loss_ref) < 1e-3 * max(1.0, abs(loss_ref))
    again = g.grad(x, d, w)
    assert again[0] == loss and np.array_equal(again[1], grad)
    g.close()
