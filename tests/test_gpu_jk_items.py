"""Fock builds on both sides of the size where work items get long (1536 quartets: n = 72 short, n = 73 long), with
run ends inside and at the ends of items, against a dense contraction in float64; several densities
at once take the same two forms.  Bound of an element: two sums of n^2 products, 2 n^2 eps times the same sums of
absolute values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 9, 40, 72, 73, 80, 81])
def test_items_short_and_long(n):
    from zinq_amd import hip
    rng = np.random.default_rng(n)
    npair = n * (n + 1) // 2
    pk = rng.standard_normal(npair * (npair + 1) // 2)
    tri = np.zeros((n, n), dtype=np.int64)
    tri[np.tril_indices(n)] = np.arange(npair)
    tri = np.maximum(tri, tri.T)
    hi, lo = np.maximum(tri[:, :, None, None], tri[None, None]), np.minimum(tri[:, :, None, None], tri[None, None])
    g = pk[hi * (hi + 1) // 2 + lo]
    H = rng.standard_normal((n, n))
    H = H + H.T
    Ps = rng.standard_normal((3, n, n))
    Ps = Ps + Ps.transpose(0, 2, 1)
    c = hip.Context(0)
    c.eri_load_packed(pk, n)
    many = c.fock_jk_multi(H, Ps)
    ga, gk = np.abs(g), g.transpose(0, 2, 1, 3).reshape(n * n, n * n)
    gka = np.abs(gk)
    for d, P in enumerate(Ps):
        # K_kl = sum_ij P_ij (ik|jl)
        ref = H + (g.reshape(n * n, n * n) @ P.ravel()).reshape(n, n) - 0.5 * (P.ravel() @ gk).reshape(n, n)
        scale = (ga.reshape(n * n, n * n) @ np.abs(P).ravel() + 0.5 * np.abs(P).ravel() @ gka).reshape(n, n)
        eps = np.finfo(float).eps
        F = c.fock_jk(H, P)
        assert np.all(np.abs(F - ref) <= 2 * n * n * eps * scale), d
        np.testing.assert_array_equal(many[d], F)
    c.close()
