"""Getters of one field called from several threads: each gets the field (they share the staging)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one piece, one value more, several pieces and a part
@pytest.mark.parametrize("n", [1 << 17, (1 << 17) + 64, 5 << 17, (5 << 17) + 320])
@pytest.mark.parametrize("precision", [32, 64])
def test_getters_from_threads(n, precision):
    import activemodelbplus.integrator as amb
    shape = (64, n // 64)
    phi = np.random.default_rng(n).standard_normal(shape, dtype=np.float32).astype(np.float64)  # exact in FP32
    sim = amb.Integrator(phi, amb.Stencil(5e-3, 1, 1), amb.Model(-0.25, 0, 0.25, 1, 0, 0, 0), precision=precision)
    np.testing.assert_array_equal(sim.field, phi)
    ens = amb.Ensemble([phi[:32], phi], amb.Stencil(5e-3, 1, 1), [amb.Model(-0.25, 0, 0.25, 1, 0, 0, 0)] * 2, [1, 2],
                       precision=precision)
    out = [None] * 4

    def get(k):
        out[k] = (sim.field, ens.field(1), sim.chemical_potential)

    threads = [threading.Thread(target=get, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for f, e, mu in out:
        np.testing.assert_array_equal(f, phi)
        np.testing.assert_array_equal(e, phi)
        np.testing.assert_array_equal(mu, out[0][2])
