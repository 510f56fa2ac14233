"""Training batches at the edges of the gradient kernel's work split: groups of 64
samples, one group per block up to two blocks per compute unit, several after
that.  Against the FP64 model with BF16-rounded operands."""
import numpy as np
import pytest

from oracle import guide as OG
from tests.test_gpu_guide import BMAX, BMIN, _batch, _dev, _features, _theta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 127, 64 * 512 - 1, 64 * 512 + 1, 64 * 1024 + 63])
def test_batch_sizes(gpu, n):
    from turner_amd.guide import Guide
    th = _theta(n % 97)
    p, nrm, w, c = _batch(n, n % 89)
    c[0] = 1.0
    args = (_dev(p), _dev(nrm), _dev(w), _dev(c))
    x = _features(p, nrm)
    lq, gq, dout = OG.loss_and_grad(th, x, w.astype(np.float64), c.astype(np.float64), quant=True)
    g = Guide(BMIN, BMAX, seed=3)
    g.set_params(th)
    loss, grad = g.loss_grad(*args)
    grad = grad.cpu().numpy().astype(np.float64)
    # An FP32 sum on the other side of a BF16 rounding boundary moves one
    # sample: its outputs by up to 3e-3, its gradient by up to 2^-8 in each of
    # the four products.
    assert abs(loss - lq) <= 1e-4 * abs(lq) + 3e-3 * np.abs(dout).sum(1).max()
    flip = 4 * 2.0 ** -8 / np.sqrt(n)
    assert np.linalg.norm(grad - gq) <= (5e-3 + flip) * np.linalg.norm(gq)
    k = 0
    for i, o in OG.LAYERS:
        for size in (o * i, o):
            sl = slice(k, k + size)
            assert np.linalg.norm(grad[sl] - gq[sl]) <= (1e-2 + flip) * np.linalg.norm(gq[sl]) + 1e-30
            k += size
    # the step from that gradient, and the operand copies it writes
    g.train_step(*args)
    new = g.params()
    ref, _, _ = OG.adam(th, grad, np.zeros_like(th), np.zeros_like(th), 1)
    d = ref - th
    assert np.all(np.abs(new - th - d) <= 2e-4 * np.abs(d) + 6e-8 * np.abs(ref) + 1e-9)
    out = g.forward(*args[:2]).cpu().numpy()
    again = Guide(BMIN, BMAX, seed=5)
    again.set_params(new)
    assert np.array_equal(out, again.forward(*args[:2]).cpu().numpy())
    again.close()
    g.close()
