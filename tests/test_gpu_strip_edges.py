"""Strips at the ends of their range: fields narrower than a strip and its halo, where noise is drawn
site by site when the columns do not split into fours, and the finite check of every kind of strip."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amb():
    import activemodelbplus.integrator as m
    return m


# one strip of 90 to 111 columns, a whole strip, two strips across fewer columns than one and its
# halos; columns 1, 2 and 3 past a multiple of four and on it
@pytest.mark.parametrize("precision,shape,temperature", [
    (32, (24000, 111), 0.05), (32, (30000, 110), 0.05), (32, (60000, 101), 0.05), (32, (30000, 112), 0.05),
    (32, (120000, 127), 0.05), (32, (30000, 107), 0.0), (64, (30000, 90), 0.05), (64, (30000, 91), 0.05),
    (64, (30000, 111), 0.0)])
def test_narrow_strips_equal_tiles(amb, precision, shape, temperature):
    """The same bits as 32x24 (FP32) or 64x16 (FP64) tiles after 5 steps."""
    rng = np.random.default_rng(shape[1])
    phi = 0.1 + 0.05 * rng.standard_normal(shape, dtype=np.float32).astype(np.float64)
    st, md = amb.Stencil(5e-3, 1.25, 0.75), amb.Model(-0.25, 0.1, 0.25, 1, 0.5, -1, temperature)
    out = []
    for tile in (0, 2):
        sim = amb.Integrator(phi, st, md, seed=3, precision=precision, tile=tile)
        assert sim.step_shape[3] == (tile == 0)
        sim.run(5)
        out.append(sim.field)
    assert np.array_equal(out[0], out[1])


# every strip kernel: quiet, noisy with and without the active current, both precisions
@pytest.mark.parametrize("precision,shape,temperature", [
    (32, (2048, 2016), 0.0), (32, (1795, 1793), 0.05), (32, (2049, 2128), 0.05), (64, (2203, 2201), 0.0),
    (64, (1399, 1401), 0.05)])
def test_strips_count_what_a_full_read_counts(amb, precision, shape, temperature):
    """Non-finite sites at a strip's and a segment's corner, on the last row and column, after two steps."""
    phi = np.full(shape, 0.1)
    phi[0, 112] = np.nan
    phi[shape[0] - 1, shape[1] - 1] = np.inf
    sim = amb.Integrator(phi, amb.Stencil(5e-3, 1, 1), amb.Model(-0.25, 0, 0.25, 1, 0.5, -1, temperature), seed=2,
                         precision=precision)
    assert sim.step_shape[3]
    with pytest.raises(amb.CudaException):
        sim.run(2)
    _, bad = sim.last_mass()
    _, bad_full = sim.mass()
    assert bad == bad_full == np.count_nonzero(~np.isfinite(sim.field)) > 2
