"""The solver's state where a solve or a setup goes wrong.

* test_nan_residuals_reset_diis: with a NaN in the right-hand side every Gram
  matrix holds NaN, which the pivot search passes over: nothing is left after
  the first pivot, the step is the plain Jacobi step and DIIS starts again.
  Spheres that do not overlap the NaN's (another molecule, 500 bohr away)
  therefore follow the plain Jacobi iteration, done here with the oracle's
  operators; 1e-11 of the iterate's size for nine steps of operators that agree
  to 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 12 spheres: DIIS and extrapolation in one launch; 600: in two
@pytest.mark.parametrize("n,lmax,ngrid", [(12, 4, 50), (600, 2, 26)])
@pytest.mark.parametrize("star", [False, True])
def test_nan_residuals_reset_diis(oracle_mod, n, lmax, ngrid, star):
    from ddpcm_amd.ddx import DDCosmo
    from ddpcm_amd.inputs import synthetic_input
    x, y, z, r = synthetic_input(n // 2, 5, lmax, ngrid).bohr()
    x, y, z, r = np.append(x, x + 500.0), np.append(y, y), np.append(z, z), np.append(r, r)
    h = DDCosmo(x, y, z, r, lmax, ngrid)
    o = oracle_mod.Oracle(x, y, z, r, lmax, ngrid)
    op = o.lstarx if star else o.lx
    facl = h.get("facl")[None, :]
    rhs = np.random.default_rng(n).standard_normal((n, h.nylm))
    rhs[0, 0] = np.nan
    got, it, ok = h.jacobi_diis(star, rhs, facl * rhs, n_iter=9)
    assert not ok and it == 10
    far = rhs.copy()
    far[:n // 2] = 0.0
    v = facl * far
    for _ in range(9):
        v = facl * (far - op(v))
    far = slice(n // 2, n)
    assert np.max(np.abs(got[far] - v[far])) <= 1e-11 * np.max(np.abs(v))
