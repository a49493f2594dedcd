"""Host arrays at the boundary: read-backs around the 1 MB chunk (n^4 doubles at n = 19 and 20 lie on both sides
of one chunk; n = 33 takes ten, past the ring of four) and multi-density Fock builds on both sides of the staged
size (1 M doubles).  The identity transform returns the ERIs, exactly the values loaded; the multi-density builds
equal the single ones bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dense(n, seed):
    """A random 8-fold symmetric <pq|rs> and its canonical packed form."""
    P = n * (n + 1) // 2
    m = np.random.default_rng(seed).standard_normal((P, P))
    m = m + m.T
    i, j = np.tril_indices(n)
    idx = np.empty((n, n), dtype=np.int64)
    idx[i, j] = idx[j, i] = np.arange(P)
    g = m[idx[:, None, :, None], idx[None, :, None, :]]  # <pq|rs> = (pr|qs)
    return np.ascontiguousarray(g), np.ascontiguousarray(m[np.tril_indices(P)])


@pytest.mark.parametrize("n", [3, 19, 20, 33])
def test_read_back_chunks(n):
    from zinq_amd import hip
    g, packed = _dense(n, n)
    with hip.Context(0) as ctx:
        ctx.eri_load_packed(packed, n)
        np.testing.assert_array_equal(ctx.ao2mo(np.eye(n)), g)
        o = n // 3 + 1
        np.testing.assert_array_equal(ctx.ao2mo(np.eye(n), o, "ovov"), g[:o, :o, o:, o:])


@pytest.mark.parametrize("nd", [2, 5348, 5352])
def test_multi_density_staging(nd):
    from zinq_amd import hip
    n = 14
    _, packed = _dense(n, 5)
    rng = np.random.default_rng(nd)
    Ps = rng.standard_normal((nd, n, n))
    Ps = Ps + Ps.transpose(0, 2, 1)
    H = Ps[0] * 0.5
    assert ((nd + 1) * n * n > 1 << 20) == (nd == 5352)
    with hip.Context(0) as ctx:
        ctx.eri_load_packed(packed, n)
        F = ctx.fock_jk_multi(H, Ps)
        for d in sorted({0, 1, nd // 2, nd - 1}):
            np.testing.assert_array_equal(F[d], ctx.fock_jk(H, Ps[d]))
