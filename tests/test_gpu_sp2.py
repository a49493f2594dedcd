"""The SP2 density of the device SCF on both sides of the size where its one-XCD form hands over to the one on all
XCDs (m = 160), from the smallest size that takes either (n = 65) on, and from several contexts at once.  Without
two-electron integrals F is the core Hamiltonian, so the density is a projector known in closed form.  Bars: the last
two steps square an eigenvalue's distance to {0, 1} (1e-9 at most before them) away, so what is left is rounding of
at most 40 steps that double it at most in their middle: 1e-10 on P, and 1e-10 n on E (second order in it)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(ctx, n, seed):
    rng = np.random.default_rng(seed)
    npair = n * (n + 1) // 2
    ctx.eri_load_packed(np.zeros(npair * (npair + 1) // 2), n)
    o = n // 5
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    w = np.concatenate([np.linspace(-20.0, -0.5, o), np.linspace(0.2, 4.0, n - o)])
    H = (Q * w) @ Q.T
    H = 0.5 * (H + H.T)
    r = ctx.scf(H, np.eye(n), 0.0, o, device=True)
    assert ctx.last_scf_driver() == "device"
    np.testing.assert_allclose(r["P"], 2.0 * Q[:, :o] @ Q[:, :o].T, rtol=0, atol=1e-10)
    assert r["E"] == pytest.approx(2.0 * w[:o].sum(), abs=1e-10 * n)


@pytest.mark.parametrize("n", [65, 80, 81, 112, 113, 144, 160, 161, 176])
def test_sp2_forms(n):
    from zinq_amd import hip
    c = hip.Context(0)
    _run(c, n, n)
    c.close()


def test_sp2_contexts_at_once():
    from zinq_amd import hip
    ctxs = [hip.Context(0) for _ in range(9)]
    errors = []

    def work(i):
        try:
            for n in (72, 100):
                _run(ctxs[i], n, 10 * n + i)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(ctxs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for c in ctxs:
        c.close()
    assert not errors, errors


def _plain_steps(F, nocc):
    """Steps plain SP2 takes on F from its Gershgorin interval: two past the first with tr X - tr X^2 < 1e-9."""
    r = np.abs(F).sum(1) - np.abs(np.diag(F))
    lo, hi = (np.diag(F) - r).min(), (np.diag(F) + r).max()
    x = np.clip((hi - np.linalg.eigvalsh(F)) / (hi - lo), 0.0, 1.0)  # the iterate's eigenvalues
    for k in range(200):
        t1, t2 = x.sum(), (x * x).sum()
        if t1 - t2 < 1e-9:
            return k + 2
        x = x * x if abs(t2 - nocc) <= abs(2 * t1 - t2 - nocc) else 2 * x - x * x
    raise AssertionError("no gap")


@pytest.mark.parametrize("guess,budget", [(40, 100), (30, 128), (2, 100)])
def test_guess_budget_below_the_iteration_budget(guess, budget):
    """The guess density and the captured iteration have step budgets of their own; a smaller one for the guess
    either is enough for it or leaves the run to the host-synchronised driver, on a fresh context in each case."""
    from zinq_amd import hip
    n, o = 70, 14
    rng = np.random.default_rng(guess)
    npair = n * (n + 1) // 2
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    w = np.concatenate([np.linspace(-20.0, -2.0, o), np.linspace(0.5, 4.0, n - o)])
    H = (Q * w) @ Q.T
    H = 0.5 * (H + H.T)
    need = _plain_steps(H, o)
    assert need <= budget and need not in (guess, guess + 1)  # away from what rounding may move
    with hip.Context(0) as c:
        c.eri_load_packed(np.zeros(npair * (npair + 1) // 2), n)
        c.set_sp2_guess_budget(guess)
        c.set_sp2_budget(budget)
        for _ in range(2):
            r = c.scf(H, np.eye(n), 0.0, o, device=True)
            assert c.last_scf_driver() == ("device" if need <= guess else "synced")
            np.testing.assert_allclose(r["P"], 2.0 * Q[:, :o] @ Q[:, :o].T, rtol=0, atol=1e-10)
            assert r["E"] == pytest.approx(2.0 * w[:o].sum(), abs=1e-10 * n)
