"""The noise paths of the fused step, against the oracle.

Interior tiles draw whole Philox groups whatever the field's column count; tiles on the
periodic seam of a field whose columns do not split into fours draw the groups that cross the
seam one site at a time.  FP64 against the FP64 oracle on the same Philox stream, 20 steps of a
field of order one: every operation rounds at 1.1e-16 and a step adds a few hundred of them
scaled by dt = 5e-3, so 1e-12 leaves three orders of margin.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amb():
    import activemodelbplus.integrator as m
    return m


# columns 1, 2 and 3 past a multiple of four; one to three tiles of 16x8 and 32x32 across, with
# and without interior tiles; the last grid has a seam tile whose last columns lie past the field
@pytest.mark.parametrize("shape", [(8, 9), (40, 61), (50, 66), (70, 131), (83, 97), (41, 35)])
def test_ragged_columns_match_oracle(amb, oracle, shape):
    st, md = (5e-3, 1.0, 1.25), (-0.25, 0.0, 0.25, 1.0, 0.5, -1.0, 0.05)
    phi = 0.05 * np.random.default_rng(shape[1]).normal(size=shape)
    ref = np.asarray(oracle.run(phi, st, md, 20, seed=11))
    for tile in range(len(amb.tile_shapes(64))):
        sim = amb.Integrator(phi, amb.Stencil(*st), amb.Model(*md), seed=11, precision=64, tile=tile + 1)
        sim.run(20)
        err = np.abs(sim.field - ref).max() / np.abs(ref).max()
        assert err < 1e-12, (shape, tile, err)


# Large fields run in strips of 112 columns and segments of rows instead of 32x32 tiles.  The
# grids have a last strip of one to 111 columns, columns that do and do not split into fours, a
# last segment shorter than the others and not a multiple of its four rows, and few rows.
@pytest.mark.parametrize("precision,shape,temperature", [
    (32, (1787, 1801), 0.0), (32, (2048, 2016), 0.0),
    (32, (1795, 1793), 0.05), (32, (2051, 2047), 0.05), (32, (2049, 2128), 0.05),
    (64, (1399, 1401), 0.05), (64, (2203, 2201), 0.0), (64, (120, 40000), 0.05)])
def test_strips_equal_tiles(amb, precision, shape, temperature):
    """The same bits as 32x24 (FP32) or 64x16 (FP64) tiles after 5 steps, and a fused mass and
    finite count equal to a full read of the field."""
    rng = np.random.default_rng(shape[0])
    phi = 0.1 + 0.05 * rng.standard_normal(shape, dtype=np.float32).astype(np.float64)
    st, md = amb.Stencil(5e-3, 1.25, 0.75), amb.Model(-0.25, 0.1, 0.25, 1, 0.5, -1, temperature)
    out = []
    for tile in (0, 2):
        sim = amb.Integrator(phi, st, md, seed=3, precision=precision, tile=tile)
        sim.run(5)
        out.append(sim.field)
        fused, bad = sim.last_mass()
        full, bad_full = sim.mass()
        # both are FP64 sums of the same values in different orders: n eps / 2 at worst, with
        # every value of order 0.1 and n = 4e6 well under 1e-9 of the sum
        assert bad == 0 and bad_full == 0 and abs(fused - full) <= 1e-9 * abs(full)
    assert np.array_equal(out[0], out[1])


def test_strips_count_nonfinite_sites(amb):
    phi = np.zeros((2048, 2050))
    phi[2047, 2049] = np.nan
    sim = amb.Integrator(phi, amb.Stencil(5e-3, 1, 1), amb.Model(-0.25, 0, 0.25, 1, 0.5, -1, 0), precision=32)
    with pytest.raises(amb.CudaException):
        sim.run(1)
    _, bad = sim.last_mass()
    _, bad_full = sim.mass()
    # L3 and G3 spread the site to a 3x3 box of mu_p and mu_a; D8 of D8 takes the box 8 sites
    # along each axis (a cross of two 3 x 19 bars), G3 of G3 to the 7x7 square, 16 sites of which
    # the cross misses
    assert bad == bad_full == (2 * 3 * 19 - 9) + 16


# Resident ensemble members that are one large tile: just past two small tiles (32 x 32 FP32,
# 32 x 16 FP64), the large tile's own size and one less, columns that do and do not split into
# fours, and members one row or column past it, which keep to small tiles.
@pytest.mark.parametrize("precision,shapes", [
    (32, [(33, 32), (32, 33), (64, 64), (63, 61), (9, 64), (64, 9), (65, 40), (30, 66)]),
    (64, [(17, 32), (16, 33), (44, 44), (48, 40), (47, 39), (9, 44), (49, 30), (30, 45)])])
def test_resident_members_equal_integrators(amb, precision, shapes):
    rng = np.random.default_rng(precision)
    st = amb.Stencil(5e-3, 1, 1.25)
    fields = [0.05 * rng.normal(size=s) for s in shapes for _ in range(2)]
    models = [amb.Model(-0.25, 0, 0.25, 1, 0.5, -1, t) for _ in shapes for t in (0.0, 0.05)]
    ens = amb.Ensemble(fields, st, models, list(range(len(fields))), precision=precision)
    assert ens.resident_count == len(fields)
    ens.run(37)  # a graph of 32 steps and a launch of five
    for i, f in enumerate(fields):
        sim = amb.Integrator(f, st, models[i], seed=i, precision=precision)
        sim.run(37)
        np.testing.assert_array_equal(ens.field(i), sim.field, err_msg=str((i, f.shape)))


# The tile of a field for which none was chosen: 32x16 tiles of 512 threads up to one round of the
# device, 32x32 tiles beyond, on one, two, four and eight XCDs, tile counts that are and are not
# multiples of eight, a last row and column of tiles that are whole, one site and partly filled.
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("shape", [(8, 9), (16, 32), (130, 127), (161, 161), (193, 200), (289, 257), (448, 450),
                                   (640, 641), (900, 868)])
def test_unchosen_tile_equals_chosen(amb, precision, shape):
    phi = 0.05 * np.random.default_rng(shape[0]).normal(size=shape)
    st = amb.Stencil(5e-3, 1, 1.25)
    for temperature in (0.0, 0.05):
        md = amb.Model(-0.25, 0, 0.25, 1, 0.5, -1, temperature)
        sims = [amb.Integrator(phi, st, md, seed=3, precision=precision, tile=tile) for tile in (0, 1)]
        for sim in sims:
            sim.run(35)  # a graph of 32 steps and three launches
        np.testing.assert_array_equal(sims[0].field, sims[1].field, err_msg=str((shape, temperature)))
        assert sims[0].last_mass()[0] == pytest.approx(sims[1].last_mass()[0], rel=1e-12, abs=1e-9)
