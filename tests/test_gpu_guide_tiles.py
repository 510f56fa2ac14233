"""The guide's network runs on tiles of 16 points, 2,048 tiles at a time, its density
on a wave per tile up to 512 x 64 points: numbers of points around these, and an
output array at an odd float, against the FP64 model
with BF16-rounded operands (bars of test_gpu_guide.py: 3e-3, and 1e-4 for 99.9%,
a single flipped rounding aside)."""
import numpy as np
import pytest

import oracle.guide as OG
from tests.test_gpu_guide import BMAX, BMIN, _batch, _dev, _features, _theta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 63, 65, 2048 * 16 - 1, 2048 * 16 + 1, 2048 * 16 * 2 + 17])
@pytest.mark.parametrize("offset", [0, 1])
def test_forward_sizes(gpu, n, offset):
    import torch
    from turner_amd import _lib
    from turner_amd.guide import Guide
    th = _theta(n % 97)
    p, nrm, w, _ = _batch(n, n % 89)
    g = Guide(BMIN, BMAX, seed=3)
    g.set_params(th)
    dp, dn = _dev(p), _dev(nrm)
    buf = torch.full((offset + n * OG.N_OUT + 7,), -77.0, device="cuda")
    _lib.check(_lib.lib().tn_guide_forward(g.handle, _lib.ptr(dp), _lib.ptr(dn), n, _lib.ptr(buf[offset:]),
                                           torch.cuda.current_stream().cuda_stream))
    buf = buf.cpu().numpy()
    assert np.all(buf[:offset] == -77.0) and np.all(buf[offset + n * OG.N_OUT:] == -77.0)
    out = buf[offset:offset + n * OG.N_OUT].reshape(n, OG.N_OUT).astype(np.float64)
    ref, _ = OG.forward(th, _features(p, nrm), quant=True)
    err = np.abs(out - ref)
    assert err.max() <= 3e-3
    assert np.count_nonzero((err > 1e-4).any(1)) <= 1 + 0.02 * n
    # the density evaluation runs the same network
    pdf = g.pdf(dp, dn, _dev(w)).cpu().numpy()
    np.testing.assert_allclose(pdf, OG.pdf(out, w.astype(np.float64)), rtol=2e-4, atol=1e-30)
    g.close()
