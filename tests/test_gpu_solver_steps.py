"""The solver's kernels at the sizes where their branches change.

* test_increment_norms_of_every_iteration: the increment norm after every
  Jacobi/DIIS iteration of both solves against the norms the reference prints
  (four digits).  The bordered system grows by a row an iteration, so a solve
  passes through every size class of its elimination (up to 8, 14, 20 and 25
  rows) and, past 24 iterations, the drop of the ten oldest vectors; a wrong
  pivot or row changes that iteration's norm and all later ones by its own
  size.  Tolerance: one unit of the last printed digit, or 5% below 1e-6 (the
  Gram dots are summed in another order, and the late increments carry that
  rounding).
"""
import numpy as np
import pytest

from conftest import deck, golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["benzene", "taxol", "l12", "crambin", "c2_small", "c2"])
def test_increment_norms_of_every_iteration(name):
    from ddpcm_amd.ddx import DDCosmo
    d, g = deck(name), golden(name)
    h = DDCosmo.from_input(d)
    h.energy_forces(d.charge)
    got = np.concatenate([h.history(0), h.history(1)])
    ref = g["residuals"]
    assert got.size == ref.size
    unit = 10.0 ** (np.floor(np.log10(ref)) - 3)
    tol = np.where(ref >= 1e-6, unit, np.maximum(unit, 5e-2 * ref))
    assert np.all(np.abs(got - ref) <= 1.01 * tol), (got, ref)
