"""Weight gradients of the surrogate over grid shapes, against the NumPy oracle.

The gradient kernels take their pixels in chunks, stages and groups that cross rows, samples
and the periodic seam differently for each shape: coarse levels of 16 and 48 columns, chunks of
several rows and of part of one, an odd number of samples.  The oracle rounds activations to
bfloat16 as the kernels do but sums in another order, and values next to a rounding edge fall
on either side (relative 2^-8 on a share of the pixels); 2e-2 in L2 per layer leaves that a
factor of several, and a pixel taken wrongly in one chunk, row or column in 64 gives more.
"""
import numpy as np
import pytest

from oracle import unet_oracle as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,n", [(64, 64, 3), (64, 192, 1), (192, 64, 1), (192, 192, 1), (64, 320, 2)])
def test_gradients_over_shapes(h, w, n):
    import activemodelbplus.integrator as amb
    rng = np.random.default_rng(h + 7 * w + n)
    S = amb.Surrogate(h, w, max_batch=n, seed=4)
    theta = S.get_params().astype(np.float64) + 0.03 * rng.normal(size=S.get_params().size)
    layout, _ = U.param_layout()
    theta[layout[0][1]:layout[0][2]].reshape(9, 32, 16)[:, :, 5:] = 0
    S.set_params(theta.astype(np.float32))
    theta = S.get_params().astype(np.float64)
    phi = rng.normal(0, 0.3, size=(n, h, w))
    params = np.stack([rng.uniform(-2, 2, n), rng.uniform(-5, 0, n), rng.uniform(-0.6, 0.6, n)], axis=1)
    target = phi + 0.05 * rng.normal(size=phi.shape)
    loss, grad = S.loss_grad(phi, params, target)
    loss_o, grad_o = U.loss_and_grad(theta, phi, params, target, emulate_bf16=True)
    assert loss == pytest.approx(loss_o, rel=2e-3)
    for name, w_off, b_off, cin, cout, taps in layout:
        for lo, hi in ((w_off, b_off), (b_off, b_off + cout)):
            if name == "head" and lo == b_off:
                continue  # telescopes to zero: a uniform current has no divergence
            err = np.linalg.norm(grad[lo:hi] - grad_o[lo:hi]) / np.linalg.norm(grad_o[lo:hi])
            assert err < 2e-2, (name, lo, err)
