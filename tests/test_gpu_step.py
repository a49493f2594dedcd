"""The one-workgroup SCF iteration (n <= 64) and its neighbour, the multi-launch form, against the CPU
oracle's SCF, at sizes on both sides of the 16-wide tile edges: n = 7, 14, 28, 35, 49, 56, 63 (one workgroup)
and 70 (multi-launch), with DIIS histories that take the register LU (up to 8), the LDS one (12) and none, and
GHF at n = 14.  Bars: the energy to 1e-10 Eh (a converged SCF's error is second order in the density error,
far below 1e-10 at the 1e-8 threshold), the orbitals as eigenvectors of the returned Fock matrix to 1e-9."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from zinq_amd import hip
    c = hip.Context(0)
    yield c
    c.close()


def _water(k):
    from zinq_amd.molecules import water_system
    s = water_system(k, basis="builtin:sto-3g")
    return s, s.hcore(), s.overlap(), s.coulomb(), s.nrep()


@pytest.mark.parametrize("k,diis", [(1, 8), (2, 8), (4, 8), (5, 3), (7, 8), (8, 12), (9, 8), (10, 8)])
def test_scf_step_sizes(ctx, k, diis):
    s, H, S, g, VN = _water(k)
    o = s.nel // 2
    ctx.eri_load_packed(s.coulomb_packed(), s.nbf)
    ro = O.scf(H, S, g, VN, o, diis=diis, threshold=1e-8)
    for fock in ("fp64", "fp32"):
        r = ctx.scf(H, S, VN, o, diis=diis, threshold=1e-8, device=True, fock_precision=fock)
        assert ctx.last_scf_driver() == "device"
        print(f"n={s.nbf} diis={diis} {fock}: dE {r['E'] - ro['E']:+.1e} it {r['iterations']}/{ro['iterations']}", flush=True)
        assert r["E"] == pytest.approx(ro["E"], abs=1e-10)
        C, e = r["C"], r["e"]
        np.testing.assert_allclose(C.T @ S @ C, np.eye(s.nbf), atol=1e-10)
        np.testing.assert_allclose(r["F"] @ C, S @ C * e, atol=1e-9)


@pytest.mark.parametrize("k", [1, 6])
def test_scf_step_without_diis(ctx, k):
    s, H, S, g, VN = _water(k)
    o = s.nel // 2
    ctx.eri_load_packed(s.coulomb_packed(), s.nbf)
    ro = O.scf(H, S, g, VN, o, diis=None, threshold=1e-8)
    r = ctx.scf(H, S, VN, o, diis=None, threshold=1e-8, device=True)
    assert ctx.last_scf_driver() == "device" and r["iterations"] == ro["iterations"]
    assert r["E"] == pytest.approx(ro["E"], abs=1e-10)


def test_scf_step_ghf(ctx):
    from zinq_amd.system import spin_block_1e, spin_block_2e
    s, H, S, g, VN = _water(1)
    Hs, Ss, gs = spin_block_1e(H), spin_block_1e(S), spin_block_2e(g)
    ctx.eri_load(gs)
    r = ctx.scf(Hs, Ss, VN, s.nel, generalized=True, device=True)
    ro = O.scf(H, S, g, VN, s.nel // 2)
    assert ctx.last_scf_driver() == "device"
    assert r["E"] == pytest.approx(ro["E"], abs=1e-10)


@pytest.mark.parametrize("n,diis", [(80, 16), (81, 3), (81, 16)])
def test_scf_launches(ctx, n, diis):
    """The multi-launch iteration with n a multiple of 16 (wide tile loads) and one above it (a last tile of one row
    and column), with short and full histories, on a positive two-electron part weak enough for SCF to settle."""
    rng = np.random.default_rng(n)
    o = n // 5
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    H = (Q * np.concatenate([np.linspace(-20.0, -2.0, o), np.linspace(0.5, 4.0, n - o)])) @ Q.T
    H = 0.5 * (H + H.T)
    S = np.eye(n) + 0.002 * (lambda a: a + a.T)(rng.standard_normal((n, n)))
    g = 0.0
    for _ in range(3):
        b = rng.standard_normal((n, n))
        b = 0.025 * (b + b.T)
        g = g + b[:, None, :, None] * b[:, None, :]
    ro = O.scf(H, S, g, 1.5, o, diis=diis, threshold=1e-8)
    ctx.eri_load(g)
    for fock in ("fp64", "fp32"):
        r = ctx.scf(H, S, 1.5, o, diis=diis, threshold=1e-8, device=True, fock_precision=fock)
        print(f"n={n} diis={diis} {fock}: dE {r['E'] - ro['E']:+.1e} it {r['iterations']}/{ro['iterations']}", flush=True)
        assert ctx.last_scf_driver() == "device"
        assert abs(r["iterations"] - ro["iterations"]) <= 1
        assert r["E"] == pytest.approx(ro["E"], abs=1e-10)


def test_scf_without_iterations_reports_its_guess(ctx):
    """A run of no iterations makes the guess density alone: one SP2 density, not folded."""
    from zinq_amd import hip
    for k in (1, 10):  # one workgroup, multi-launch
        s, H, S, g, VN = _water(k)
        ctx.eri_load_packed(s.coulomb_packed(), s.nbf)
        with pytest.raises(hip.ScfDidNotConverge):
            ctx.scf(H, S, VN, s.nel // 2, iterations=0, device=True)
        sp2 = ctx.last_scf_sp2()
        assert ctx.last_scf_driver() == "device" and ctx.scf_replays() == 0
        assert sp2["densities"] == 1 and sp2["folded"] == 0 and sp2["steps"] > 1, sp2


def test_scf_history_beyond_the_device(ctx):
    """A DIIS history above 16 goes to the host-synchronised driver at once, on the inputs set up before it."""
    s, H, S, g, VN = _water(5)
    o = s.nel // 2
    ctx.eri_load_packed(s.coulomb_packed(), s.nbf)
    ro = O.scf(H, S, g, VN, o, diis=20, threshold=1e-8)
    r = ctx.scf(H, S, VN, o, diis=20, threshold=1e-8, device=True)
    assert ctx.last_scf_driver() == "synced" and r["iterations"] == ro["iterations"]
    assert r["E"] == pytest.approx(ro["E"], abs=1e-10)


def test_batch_largest_molecules():
    """Batch molecules on five and six tiles (n = 73 .. 96) with a two-electron part, in a batch that was not
    autotuned, so that their Fock builds take long work items, beside a small molecule in the short form and alone in the
    long one, and again after the autotuner chose: the oracle's SCF to the bars above, alone and mixed the same bits."""
    from zinq_amd.batch import Batch
    mols = []
    for n in (7, 73, 80, 81, 96):
        rng = np.random.default_rng(n)
        o = max(1, n // 5)
        Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        H = (Q * np.concatenate([np.linspace(-20.0, -2.0, o), np.linspace(0.5, 4.0, n - o)])) @ Q.T
        S = np.eye(n) + 0.002 * (lambda a: a + a.T)(rng.standard_normal((n, n)))
        tri = np.tril_indices(n)
        m = 0.0
        for _ in range(3):  # (pq|rs) = sum of b_pq b_rs
            b = rng.standard_normal((n, n))
            b = 0.025 * (b + b.T)[tri]
            m = m + b[:, None] * b[None, :]
        mols.append((0.5 * (H + H.T), S, 1.5, o, m[np.tril_indices(len(b))]))
    ref = [O.scf(H, S, None, VN, o, threshold=1e-8, packed=pk) for H, S, VN, o, pk in mols]
    mix = Batch(0)
    for m in mols:
        mix.add(*m)
    for tuned in (False, True):
        if tuned:
            print("autotuned:", mix.autotune(), flush=True)
        r = mix.run(threshold=1e-8)
        assert (r["status"] == 0).all(), r["status"]
        for k, ro in enumerate(ref):
            print(f"n={len(mols[k][0])} tuned={tuned}: dE {r['E_rhf'][k] - ro['E']:+.1e} it {r['iterations'][k]}/"
                  f"{ro['iterations']}", flush=True)
            assert r["E_rhf"][k] == pytest.approx(ro["E"], abs=1e-10)
            assert abs(r["iterations"][k] - ro["iterations"]) <= 1
            if not tuned:
                alone = Batch(0)
                alone.add(*mols[k])
                ra = alone.run(threshold=1e-8)
                assert ra["E_rhf"][0] == r["E_rhf"][k] and ra["E_corr"][0] == r["E_corr"][k]
                assert ra["iterations"][0] == r["iterations"][k]
                alone.close()
    mix.close()
