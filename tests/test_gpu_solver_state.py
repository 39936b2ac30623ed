"""The solver's state where a solve or a setup goes wrong.

* test_nan_residuals_reset_diis: with a NaN in the right-hand side every Gram
  matrix holds NaN, which the pivot search passes over: nothing is left after
  the first pivot, the step is the plain Jacobi step and DIIS starts again.
  Spheres that do not overlap the NaN's (another molecule, 500 bohr away)
  therefore follow the plain Jacobi iteration, done here with the oracle's
  operators; 1e-11 of the iterate's size for nine steps of operators that agree
  to 1e-12.
* test_failed_setup_is_refused: after a geometry whose setup failed (a sphere
  with more than 64 neighbours) every call that walks the setup's lists, which
  are half made then, is refused; the sizes and the last results stay; the next
  good geometry gives a fresh handle's results, bit for bit.
* test_solve_records: solves of different lengths in turn on one handle, so that a
  value read from the record of the solve before would show: iteration counts,
  flags and all norms equal those of the same solve made first.
* test_two_launch_solver_equals_batch_of_two, test_two_launch_solver_short_histories:
  single systems whose DIIS and extrapolation are two latency-ordered launches
  (more spheres than two a compute unit; the extrapolation's launches are
  counted, so that a size that takes another path fails).  Both solutions equal
  the general kernels', which a batch takes, bit for bit (a sweep worker has at
  most one unit at these sizes, so the operators' sums are split alike), at one
  and several elements a thread.  14 points do not resolve lmax 6 and 16: there
  the iteration, the reference's too, wanders on, and the iterates after all 200
  steps are compared, past many drops of the oldest vectors.  Shorter histories, whose later slots do not
  exist, give the same solution (1e-10 in the h^-1/2 norm for increments below
  1e-12).
"""
import ctypes as C

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


@pytest.mark.parametrize("batch", [False, True])
def test_failed_setup_is_refused(batch):
    from ddpcm_amd.ddx import DDCosmo, DDCosmoBatch, DDXError
    from ddpcm_amd.inputs import synthetic_input
    n = 80
    d = synthetic_input(n, 3, 4, 50)
    x, y, z, r = d.bohr()
    q = d.charge
    copies = 2 if batch else 1

    def new():
        if batch:
            return DDCosmoBatch([x] * 2, [y] * 2, [z] * 2, [r] * 2, 4, 50)
        return DDCosmo(x, y, z, r, 4, 50)

    def upload(v, scale):
        v.upload(*[np.tile(a, copies) for a in (scale * x, scale * y, scale * z, r, q)])

    h = new()
    upload(h, 1.0)
    h.run()
    before = h.result()
    sigma = h.get("sigma")
    v = np.ones((copies * n, h.nylm))
    cav = np.zeros(h.ncav)
    upload(h, 0.01)   # all spheres within one another: 79 neighbours each
    with pytest.raises(DDXError) as e:
        h.run()
    assert e.value.code == 4
    calls = [lambda: h.lx(v), lambda: h.lstarx(v), lambda: h.mkrhs(np.tile(q, copies)),
             lambda: h.forces_dd(cav, v, v), lambda: h.ddmkzeta(v), lambda: h.neighbours(),
             lambda: h.guess_train(1)]
    calls += [lambda a=a: h.get(a) for a in ("fi", "ui", "zi", "ccav")]
    if not batch:
        calls += [lambda: h.cosmo(False, phi=cav, psi=v), lambda: h.cosmo(True, psi=v),
                  lambda: h.jacobi_diis(False, v, v)]
    for call in calls:
        with pytest.raises(DDXError) as e:
            call()
        assert e.value.code == 6 and "setup" in str(e.value)
    with pytest.raises(DDXError) as e:   # sets up again, and meets the same error
        h.energy_forces([q] * 2 if batch else q)
    assert e.value.code == 4
    h.stats()
    for old, now in zip(before, h.result()):
        assert np.array_equal(old, now)
    assert np.array_equal(sigma, h.get("sigma"))
    if batch:
        off = np.zeros(3, dtype=np.int32)
        h._check(h.L.ddx_batch_sizes(h.h, None, None, off.ctypes.data_as(C.POINTER(C.c_int))))
        assert np.array_equal(off, h.cav_off)
    upload(h, 1.01)
    h.run()
    f = new()
    upload(f, 1.01)
    f.run()
    for a, b in zip(h.result(), f.result()):
        assert np.array_equal(a, b)
    assert np.array_equal(h.lx(v), f.lx(v))


def test_solve_records():
    from ddpcm_amd.ddx import DDCosmo
    from ddpcm_amd.inputs import synthetic_input
    x, y, z, r = synthetic_input(20, 8, 2, 26).bohr()
    h = DDCosmo(x, y, z, r, 2, 26)
    rhs = np.random.default_rng(2).standard_normal((20, h.nylm))
    x0 = h.get("facl")[None, :] * rhs

    def solve(star, tol, cap):
        _, it, ok = h.jacobi_diis(star, rhs, x0, tol=tol, n_iter=cap)
        return it, ok, h.history(star)

    kinds = [(star, tol, cap) for star in (0, 1)
             for tol, cap in ((1e-12, 200), (1e-2, 200), (1e-12, 3), (1e-6, 200))]
    first = [solve(*k) for k in kinds]
    assert len({f[0] for f in first}) >= 4
    for it, ok, hist in first:
        assert hist.size == (it if ok else it - 1)
    rng = np.random.default_rng(4)
    for k in rng.integers(len(kinds), size=300):
        it, ok, hist = solve(*kinds[k])
        assert (it, ok) == first[k][:2] and np.array_equal(hist, first[k][2])


def _two_launches(h):
    """Whether the solve just timed had launches of the extrapolation alone."""
    return h.kernel_timer_read("extrap")[0] > 0


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("n,lmax,ngrid", [(601, 0, 26), (600, 2, 26), (901, 6, 14), (700, 16, 14)])
def test_two_launch_solver_equals_batch_of_two(n, lmax, ngrid, mixed):
    from ddpcm_amd.ddx import DDCosmo, DDCosmoBatch, NotConverged
    from ddpcm_amd.inputs import synthetic_input
    d = synthetic_input(n, 77 + n, lmax, ngrid)
    x, y, z, r = d.bohr()
    h = DDCosmo(x, y, z, r, lmax, ngrid)
    b = DDCosmoBatch([x, x], [y, y], [z, z], [r, r], lmax, ngrid)
    for v in (h, b):
        v.set_precision(mixed)
    h.kernel_timer("extrap")
    converged = lmax < 6
    for v, q in ((h, d.charge), (b, [d.charge, d.charge])):
        if converged:
            v.energy_forces(q)
        else:
            with pytest.raises(NotConverged):
                v.energy_forces(q)
    assert _two_launches(h)
    for name in ("sigma", "s"):
        one, two = h.get(name), b.get(name)
        assert np.all(np.isfinite(one))
        assert np.array_equal(one, two[:n]) and np.array_equal(one, two[n:]), name


@pytest.mark.parametrize("star", [False, True])
@pytest.mark.parametrize("n,lmax,ngrid", [(600, 2, 26), (1300, 6, 110)])
def test_two_launch_solver_short_histories(n, lmax, ngrid, star):
    from ddpcm_amd.ddx import DDCosmo
    from ddpcm_amd.inputs import synthetic_input
    x, y, z, r = synthetic_input(n, 5 + n, lmax, ngrid).bohr()
    h = DDCosmo(x, y, z, r, lmax, ngrid)
    rhs = np.random.default_rng(n).standard_normal((n, h.nylm))
    x0 = h.get("facl")[None, :] * rhs
    ref, _, ok = h.jacobi_diis(star, rhs, x0, tol=1e-12)
    assert ok
    h.kernel_timer("extrap")
    for m in (11, 12, 18, 24):
        got, _, ok = h.jacobi_diis(star, rhs, x0, diis_max=m, tol=1e-12)
        assert _two_launches(h)
        assert ok and h.hnorm(got - ref) <= 1e-10, m
