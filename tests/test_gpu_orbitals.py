"""Orbitals of a batch: the in-LDS Jacobi eigenpairs against scipy's generalized eigh at the edges of its lane
widths (32, 64) and of its range (2, 96), odd sizes, and with degenerate eigenvalues."""

import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _no_interaction(n, seed, degenerate=False):
    """H and S of n functions; without two-electron integrals the converged F is H."""
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n)) * 0.3 / np.sqrt(n)
    S = np.eye(n) + 0.5 * (A + A.T)
    if degenerate:  # threefold levels, H = S V diag V^T S with V^T S V = 1
        V = np.linalg.inv(np.linalg.cholesky(S)).T @ np.linalg.qr(rng.standard_normal((n, n)))[0]
        e = -8.0 + np.arange(n) // 3
        H = S @ (V * e) @ V.T @ S
    else:
        B = rng.standard_normal((n, n))
        H = 0.2 * (B + B.T) + np.diag(np.linspace(-20.0, 3.0, n))
    return 0.5 * (H + H.T), S


@pytest.mark.parametrize("degenerate", [False, True])
def test_batch_orbitals_vs_scipy(degenerate):
    from zinq_amd.batch import Batch

    sizes = [2, 3, 5, 6, 7, 31, 32, 33, 63, 64, 65, 95, 96]
    b = Batch(0)
    mats = []
    for n in sizes:
        H, S = _no_interaction(n, 100 + n, degenerate)
        npair = n * (n + 1) // 2
        # an occupied space that ends between levels of the degenerate spectrum
        nocc = max(1, n // 2 // 3 * 3) if degenerate else max(1, n // 3)
        b.add(H, S, 0.0, min(nocc, n - 1), np.zeros(npair * (npair + 1) // 2))
        mats.append((H, S))
    r = b.run(iterations=50)
    for k, (H, S) in enumerate(mats):
        n = len(S)
        if not degenerate:
            assert r["status"][k] == 0, n
        e, C = b.orbitals(k)
        w = scipy.linalg.eigh(H, S, eigvals_only=True)
        # rounding of a backward stable solver, n eps |S^-1 H|, with a factor 16 for forming F' and S^-1/2
        scale = np.abs(w).max() * np.linalg.cond(S)
        tol = 16 * n * EPS * scale
        assert np.all(np.diff(e) >= 0), n
        np.testing.assert_allclose(e, w, rtol=0, atol=tol, err_msg=str(n))
        np.testing.assert_allclose(C.T @ S @ C, np.eye(n), rtol=0, atol=16 * n * EPS * np.linalg.cond(S), err_msg=str(n))
        np.testing.assert_allclose(H @ C, S @ C * e, rtol=0, atol=tol * np.abs(S).sum(1).max() * np.abs(C).max(), err_msg=str(n))
    b.close()


@pytest.mark.parametrize("n", [6, 33, 70])
def test_batch_orbitals_zero_levels(n):
    """Levels at zero that couplings of 1e-20 to a low level split by 1e-41 of the largest element: a gap and a pivot
    below the range of normal single-precision numbers.  The matrix is diagonal to working precision, so the
    levels come back to n eps of the largest and the orbitals orthonormal to n eps."""
    from zinq_amd.batch import Batch

    nocc, zeros = 2, n // 2
    w = np.concatenate([[-8.0, -4.0], np.zeros(zeros), np.linspace(1.0, 3.0, n - 2 - zeros)])
    H = np.diag(w)
    H[0, 2:2 + zeros] = H[2:2 + zeros, 0] = 1e-20 * np.arange(1, zeros + 1)
    npair = n * (n + 1) // 2
    b = Batch(0)
    b.add(H, np.eye(n), 0.0, nocc, np.zeros(npair * (npair + 1) // 2))
    r = b.run(iterations=50)
    e, C = b.orbitals(0)
    b.close()
    assert r["status"][0] == 0
    np.testing.assert_allclose(e, w, rtol=0, atol=16 * n * EPS * 8.0)
    np.testing.assert_allclose(C.T @ C, np.eye(n), rtol=0, atol=16 * n * EPS)
