"""The network's gradients at rows around the weight gradient's 16-cell pieces
and grids of one to several pieces a wave, as test_gradients_match_reference
checks them at one shape (BF16 operands: 3e-2 relative, cosine 0.999)."""
import numpy as np
import pytest

from pllcart3d_amd import closure as CL

from test_gpu_closure import R, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 4, 15), (4, 5, 17), (3, 6, 33), (24, 16, 31), (40, 20, 48)])
def test_gradient_at_piece_edges(shape):
    rng, Pd, x5, x, net = _setup(shape, 2)
    t = rng.normal(size=shape)
    mask = (rng.uniform(size=shape) > 0.2).astype(np.uint8)
    L, g = net.loss_grad(net.add_sample(x5, t, mask))
    Lr, Gr, _ = R.loss_and_grads(x, t, mask.astype(bool), Pd)
    gr = CL.flat_from_dict({k: Gr[k] for k in Gr})
    w = 27 * 256
    for q in range(3):
        for sl in (slice(q * (w + 16), q * (w + 16) + w), slice(q * (w + 16) + w, (q + 1) * (w + 16))):
            a, b = g[sl], gr[sl]
            e = np.linalg.norm(a - b) / np.linalg.norm(b)
            assert e <= 3e-2 and a @ b >= 0.999 * np.linalg.norm(a) * np.linalg.norm(b), (shape, q, sl, e)
    net.close()
