"""zq_eigh at the edges of its two tridiagonal reductions (n <= 32 and up to 192) and of the wide one's stages of
32, and on matrices whose rows vanish or whose elements are large: eigenvalues against LAPACK's, U^T U = 1 and
A U = U W.  Tolerances: a backward stable solver leaves n eps |A|, taken with a factor 16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def ctx():
    from zinq_amd import hip
    c = hip.Context(0)
    yield c
    c.close()


def _matrix(n, kind):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A = A + A.T
    if kind == "blocks":  # two blocks and a zero row: reflectors without a tail
        h = n // 2
        A[:h, h:] = A[h:, :h] = 0.0
        A[h, :] = A[:, h] = 0.0
    elif kind == "tridiagonal":  # every tail zero
        A = np.triu(np.tril(A, 1), -1)
    elif kind == "large":
        A *= 1e140
    return A


@pytest.mark.parametrize("kind", ["plain", "blocks", "tridiagonal", "large"])
@pytest.mark.parametrize("n", [31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 160, 161, 191, 192])
def test_reduction_edges(ctx, n, kind):
    A = _matrix(n, kind)
    W, U = ctx.eigh(A)
    w = np.linalg.eigvalsh(A)
    tol = 16 * n * EPS * np.abs(w).max()
    np.testing.assert_allclose(W, w, rtol=0, atol=tol)
    np.testing.assert_allclose(U.T @ U, np.eye(n), rtol=0, atol=16 * n * EPS)
    np.testing.assert_allclose(A @ U, U * W, rtol=0, atol=tol)
