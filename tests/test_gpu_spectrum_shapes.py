"""Binned spectrum over grid shapes against NumPy.

A wave bins 64 modes of the half spectrum at a time by runs of equal bins: narrow grids put many
rows in a wave, wide ones part of one, and coarse edges make runs of a whole row.  FP64: the FFTs
agree to about log2(n) 1e-16 of the largest mode and a bin's sum has fewer than 1e5 terms, so
1e-11 of the total leaves two orders; counts are equal because no |k| falls on an edge (edges are
offset by 0.37 of a mode; distinct |k|^2 in units of the smallest mode differ by far more than
rounding).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 9), (9, 64), (33, 130), (130, 126), (257, 129), (8, 1024)])
@pytest.mark.parametrize("nedges", [1, 5, 300])
def test_binned_spectrum_matches_numpy(shape, nedges):
    import activemodelbplus.integrator as amb
    ny, nx = shape
    phi = 0.1 * np.random.default_rng(ny + nx).normal(size=shape)
    sim = amb.Integrator(phi, amb.Stencil(5e-3, 1, 1), amb.Model(-0.25, 0, 0.25, 1, 0, 0, 0), precision=64)
    edges = (np.arange(nedges) + 0.3711) * (np.pi * 1.4 / nedges)
    sums, counts = sim.structure_factor_bins(edges)
    power = np.abs(np.fft.fft2(phi - phi.mean())) ** 2
    ky, kx = (np.fft.fftfreq(n) * 2 * np.pi for n in shape)
    where = np.digitize(np.sqrt(ky[:, None] ** 2 + kx[None, :] ** 2), edges, right=True).ravel()
    np.testing.assert_array_equal(counts, np.bincount(where, minlength=nedges + 1))
    ref = np.bincount(where, power.ravel(), minlength=nedges + 1)
    assert np.abs(sums - ref).max() < 1e-11 * power.sum()
