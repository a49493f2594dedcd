"""The first quarter transform at the edges of its layouts: one block and odd numbers of blocks, occupied counts on
both sides of its 16-column tiles, against the transform in float64.  Bound of an element: four chained sums of n
products each, 4 n eps times the same transform of the absolute values (eps of the element type, once more for
rounding the integrals and coefficients to it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from zinq_amd import hip
    c = hip.Context(0)
    yield c
    c.close()


def _ovov(g, C, o):
    X = np.einsum("mnls,mi->inls", g, C[:, :o], optimize=True)
    X = np.einsum("inls,lj->ijns", X, C[:, :o], optimize=True)
    X = np.einsum("ijns,na->ijas", X, C[:, o:], optimize=True)
    return np.einsum("ijas,sb->ijab", X, C[:, o:], optimize=True)


@pytest.mark.parametrize("n,o", [(3, 1), (8, 7), (9, 1), (17, 15), (17, 16), (41, 16), (41, 17), (41, 31), (41, 33), (40, 39),
                                 (57, 48), (58, 49)])
def test_first_quarter_edges(ctx, n, o):
    rng = np.random.default_rng(100 * n + o)
    np_ = n * (n + 1) // 2
    pk = rng.standard_normal(np_ * (np_ + 1) // 2)
    tri = np.zeros((n, n), dtype=int)
    tri[np.tril_indices(n)] = np.arange(np_)
    tri = np.maximum(tri, tri.T)
    I, J = tri[:, :, None, None], tri[None, None]
    hi, lo = np.maximum(I, J), np.minimum(I, J)
    g = pk[hi * (hi + 1) // 2 + lo]
    C = rng.standard_normal((n, n)) / np.sqrt(n)
    ctx.eri_load_packed(pk, n)
    ref, scale = _ovov(g, C, o), _ovov(np.abs(g), np.abs(C), o)
    for precision, eps in (("fp64", np.finfo(np.float64).eps), ("fp32", np.finfo(np.float32).eps), ("fp32c", np.finfo(np.float32).eps)):
        out = ctx.ao2mo(C, o, "ovov", precision=precision)
        assert np.all(np.abs(out - ref) <= (4 * n + 8) * eps * scale), (n, o, precision)


@pytest.mark.parametrize("n,o", [(2, 1), (9, 8), (33, 16), (34, 17), (41, 20), (58, 25), (75, 11)])
def test_group_takes_the_same_path(n, o):
    """A batch's MP2 is zq_mp2 of its orbitals to the last bit in every precision: odd and even numbers of virtuals
    (the register-direct Q3 and Q4 take pairs of them, or one at a time), one to four tiles of them."""
    from zinq_amd import hip
    from zinq_amd.batch import Batch
    rng = np.random.default_rng(n + o)
    np_ = n * (n + 1) // 2
    pk = 1e-3 * rng.standard_normal(np_ * (np_ + 1) // 2)  # small: the SCF is that of H
    H = np.diag(np.concatenate([np.linspace(-9.0, -3.0, o), np.linspace(1.0, 5.0, n - o)]))
    for precision in ("fp64", "fp32", "fp32c"):
        b = Batch(0)
        b.add(H, np.eye(n), 0.0, o, pk)
        r = b.run(mp2_precision=precision)
        e, C = b.orbitals(0)
        b.close()
        c = hip.Context(0)
        c.eri_load_packed(pk, n)
        assert r["status"][0] == 0
        assert r["E_corr"][0] == c.mp2(C, e, o, precision=precision), precision
        c.close()


@pytest.mark.parametrize("n,o", [(121, 8), (128, 17), (129, 8), (136, 17), (145, 18)])
def test_last_quarters_both_forms(ctx, n, o):
    """Q3 and Q4 of the 4-byte forms on both sides of the size (128 padded functions) where they go from registers to
    tiles in LDS; integrals of rank 2, so that the reference needs no dense tensor."""
    rng = np.random.default_rng(n + o)
    B = rng.standard_normal((2, n, n))
    B = B + B.transpose(0, 2, 1)
    low = np.tril_indices(n)
    b = B[:, low[0], low[1]]
    pk = np.concatenate([b[:, t] @ b[:, :t + 1] for t in range(b.shape[1])])
    C = rng.standard_normal((n, n)) / np.sqrt(n)
    ctx.eri_load_packed(pk, n)

    M, A = (np.einsum("mi,pmn,na->pia", c[:, :o], x, c[:, o:], optimize=True) for x, c in ((B, C), (np.abs(B), np.abs(C))))
    ref, scale = np.einsum("pia,pjb->ijab", M, M), np.einsum("pia,pjb->ijab", A, A)
    for precision in ("fp64", "fp32", "fp32c"):
        out = ctx.ao2mo(C, o, "ovov", precision=precision)
        eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
        assert np.all(np.abs(out - ref) <= (4 * n + 8) * eps * scale), (n, o, precision)
