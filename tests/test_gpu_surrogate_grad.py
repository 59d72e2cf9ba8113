"""Gradients of the surrogate over grid shapes: translating a sample must not change them.

The gradient kernels take their pixels in chunks, stages and segments that cross rows, samples
and the periodic seam differently for each shape and batch: coarse levels of 16 and 48 columns,
chunks of several rows and of part of one.  A translation by multiples of four moves every
activation and gradient image exactly (pooling keeps its phase), so the gradient of a sample and
that of a batch of it and its translate (whose mean halves exactly) are the same terms summed in
another order and other chunks.  The terms of a parameter's N <= 122880 pixels vary in sign, so a
partial sum is about sqrt(N) terms large and N roundings of 2^-24 of that add up to
sqrt(N) 2^-24 = 2e-5 of the sum; 1e-3 leaves a factor of fifty, and one row, column or chunk of
pixels taken wrongly gives several times that.  Values against the oracle: test_gpu_surrogate.py.
"""
import numpy as np
import pytest

from oracle import unet_oracle as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,shift", [(64, 64, (20, 12)), (64, 192, (4, 100)), (192, 64, (100, 28)),
                                       (192, 192, (64, 8)), (64, 320, (32, 300)), (256, 256, (252, 4))])
def test_translated_sample_has_the_same_gradient(h, w, shift):
    import activemodelbplus.integrator as amb
    rng = np.random.default_rng(h + 7 * w)
    S = amb.Surrogate(h, w, max_batch=2, seed=4)
    theta = S.get_params()
    S.set_params((theta + 0.03 * rng.normal(size=theta.size)).astype(np.float32))
    phi = rng.normal(0, 0.3, size=(1, h, w))
    params = np.array([[0.5, -2.0, 0.3]])
    target = phi + 0.05 * rng.normal(size=phi.shape)
    pair = [np.concatenate([a, np.roll(a, shift, axis=(1, 2))]) for a in (phi, target)]
    loss, grad = S.loss_grad(phi, params, target)
    loss2, grad2 = S.loss_grad(pair[0], np.repeat(params, 2, axis=0), pair[1])
    assert loss2 == pytest.approx(loss, rel=1e-5)
    layout, _ = U.param_layout()
    for name, w_off, b_off, cin, cout, taps in layout:
        for lo, hi in ((w_off, b_off), (b_off, b_off + cout)):
            if name == "head" and lo == b_off:
                continue  # telescopes to zero: a uniform current has no divergence
            err = np.linalg.norm(grad2[lo:hi] - grad[lo:hi]) / np.linalg.norm(grad[lo:hi])
            assert err < 1e-3, (name, lo, err)
