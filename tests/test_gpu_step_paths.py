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
