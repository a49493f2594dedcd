"""Performance cases: the calls a user of zinq_amd makes, over the sizes they make them at.

Every pass goes through the public Python entry points (zinq_amd.hip.Context, zinq_amd.batch.Batch),
which are the C ABI's calls one to one: host arrays in, host arrays out, with a molecule's ERIs resident
on the device, as an SCF driver, a response solver, a correlation method or a serving loop keeps them.

Two kinds of input:
- single calls (Fock builds, transforms, MP2, eigensolves) run on the exact ERIs of n normalised s
  Gaussians at random places in a box that grows with n, exponents 0.15 .. 20, so that magnitudes and
  decay are those of a molecule in a small basis; they are made on the GPU in milliseconds;
- whole SCF runs and the batch need a molecule that converges: water clusters with distorted monomers,
  integrals from the package's own host engine.
"""
import math

import numpy as np
import torch

from zinq_amd import hip
from zinq_amd.batch import Batch
from zinq_amd.molecules import batch_specs, batch_system, water_system

# Occupied orbitals of a closed-shell molecule with n basis functions: water has 5 of 24 in cc-pVDZ.
OCC_SHARE = 5.0 / 24.0


def listed():
    return [
        # one Fock build per SCF iteration of a driver that keeps its own loop (getFock): a single water,
        # cc-pVDZ, where the call's fixed costs are all there is ...
        dict(name="fock_24", op="fock", n=24, x=0.5),
        # ... and eight waters, where the ERIs stream from HBM
        dict(name="fock_192", op="fock", n=192, x=0.5),
        # CPHF: the response densities of six perturbations in one pass, ragged size (not a multiple of 8)
        dict(name="multi_93x6", op="multi", n=93, nd=6, x=0.5),
        # the (ia|jb) block handed back to a host method, ragged sizes
        dict(name="ovov_75", op="ao2mo", n=75, o=16, block="ovov"),
        # all MO integrals of a small molecule, as CI and higher MPn need them
        dict(name="full_41", op="ao2mo", n=41, o=0, block="full"),
        # MP2 correlation energies: eight waters in FP64, and the serving path's FP32 products with FP64
        # sums at an odd size
        dict(name="mp2_192_fp64", op="mp2", n=192, o=40, precision="fp64"),
        dict(name="mp2_101_fp32c", op="mp2", n=101, o=21, precision="fp32c"),
        # eigenpairs of an orthonormal-basis Fock matrix
        dict(name="eigh_150", op="eigh", n=150),
        # whole device SCF runs with the interface's default options: one water, six waters; and the
        # serving loop's mixed path for four waters
        dict(name="scf_water1", op="scf", k=1, basis="cc-pvdz", spacing=3.0, mixed=False),
        dict(name="scf_water6", op="scf", k=6, basis="cc-pvdz", spacing=3.0, mixed=False),
        dict(name="scf_water4_mixed", op="scf", k=4, basis="cc-pvdz", spacing=3.0, mixed=True),
        # many small molecules of uneven size at once, RHF + MP2
        dict(name="batch_96", op="batch", count=96),
    ]


def draw(rng):
    """One more case of the same kinds and ranges."""

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["fock", "fock", "multi", "ao2mo", "mp2", "mp2", "eigh", "scf", "scf", "batch"])
    if op == "fock":
        return dict(op=op, n=size(7, 192), x=rng.choice([0.5, 0.5, 1.0]))
    if op == "multi":
        return dict(op=op, n=size(7, 128), nd=rng.randint(2, 9), x=rng.choice([0.5, 1.0]))
    if op == "ao2mo":
        if rng.random() < 0.5:
            return dict(op=op, n=size(7, 48), o=0, block="full")
        n = size(12, 96)
        return dict(op=op, n=n, o=max(1, min(n - 1, int(n * rng.uniform(0.12, 0.4)))), block="ovov")
    if op == "mp2":
        n = size(12, 192)
        return dict(op=op, n=n, o=max(1, min(n // 4, int(n * rng.uniform(0.12, 0.25)))),
                    precision=rng.choice(["fp64", "fp64", "fp32c", "fp32"]))
    if op == "eigh":
        return dict(op=op, n=size(7, 320))
    if op == "scf":
        d = dict(op=op, spacing=round(rng.uniform(2.9, 3.4), 3))  # lattice spacing of the cluster, Angstrom
        if rng.random() < 0.3:
            return dict(d, k=rng.randint(1, 8), basis="sto-3g", mixed=False)
        return dict(d, k=rng.randint(1, 6), basis="cc-pvdz", mixed=rng.random() < 0.5)
    return dict(op=op, count=rng.randint(8, 96))


# ---------------------------------------------------------------------------------------------- inputs


def _generator(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + case["n"])
    return g


def _pair_eris(n, g):
    """(ij|kl) over pairs i >= j, k >= l of normalised s Gaussians, as the full npair x npair matrix on the
    GPU, and the overlap matrix: (ij|kl) = S_ij S_kl erf(sqrt(rho) R) / R."""
    f64 = dict(dtype=torch.float64, device="cuda")
    side = 5.7 * max(1.0, n / 24.0) ** (1.0 / 3.0)
    at = torch.rand((n, 3), generator=g, **f64) * side
    a = torch.exp(torch.rand(n, generator=g, **f64) * math.log(20.0 / 0.15)) * 0.15
    i, j = torch.tril_indices(n, n, device="cuda")
    p = a[i] + a[j]
    r2 = (at[i] - at[j]).square().sum(1)
    s = (2.0 * torch.sqrt(a[i] * a[j]) / p) ** 1.5 * torch.exp(-a[i] * a[j] / p * r2)
    mid = (a[i, None] * at[i] + a[j, None] * at[j]) / p[:, None]
    m = torch.empty((p.numel(), p.numel()), **f64)
    for c in range(0, p.numel(), 2048):
        e = slice(c, c + 2048)
        rho = p[e, None] * p[None] / (p[e, None] + p[None])
        d2 = torch.zeros_like(rho)
        for x in range(3):
            d2 += (mid[e, x, None] - mid[None, :, x]).square()
        d = torch.sqrt(d2)
        near = 2.0 / math.sqrt(math.pi) * torch.sqrt(rho)  # the limit at d = 0
        v = torch.where(d > 1e-7, torch.erf(torch.sqrt(rho) * d) / d.clamp_min(1e-7), near)
        m[e] = v * s[e, None] * s[None]
    m = torch.tril(m) + torch.tril(m, -1).T  # exactly symmetric
    S = torch.empty((n, n), **f64)
    S[i, j] = s
    S[j, i] = s
    return m, S


def _pack(m):
    """Canonical packed ERIs (row I = pair i >= j, columns J <= I) as a host array."""
    keep = torch.ones(m.shape, dtype=torch.bool, device=m.device).tril_()
    return m[keep].cpu().numpy()


def _orbitals(n, g):
    """An orthonormal set of orbitals (columns) and their energies with a gap."""
    q, _ = torch.linalg.qr(torch.randn((n, n), generator=g, dtype=torch.float64, device="cuda"))
    return q


def _energies(n, o, g):
    lo = -0.4 - 20.0 * torch.rand(o, generator=g, dtype=torch.float64, device="cuda") ** 3
    hi = 0.1 + 4.0 * torch.rand(n - o, generator=g, dtype=torch.float64, device="cuda")
    return torch.cat([lo.sort().values, hi.sort().values])


def _core(S, g):
    """A core-Hamiltonian-like symmetric matrix: attraction in proportion to the overlap."""
    z = 1.0 + 7.0 * torch.rand(S.shape[0], generator=g, dtype=torch.float64, device="cuda")
    return -0.5 * S * (z[:, None] + z[None])


def _densities(n, o, count, g):
    q = [torch.linalg.qr(torch.randn((n, o), generator=g, dtype=torch.float64, device="cuda"))[0] for _ in range(count)]
    return torch.stack([2.0 * c @ c.T for c in q])


def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


def _single(case, seed):
    """The device tensors of a single-call case, in a fixed order of draws."""
    n, op = case["n"], case["op"]
    g = _generator(case, seed)
    d = {}
    if op == "eigh":
        # orthonormal-basis Fock matrix: core, valence and virtual levels in a rotated basis
        q = _orbitals(n, g)
        e = _energies(n, max(1, int(n * OCC_SHARE)), g)
        f = (q * e) @ q.T
        d["A"] = 0.5 * (f + f.T)
        return d
    d["m"], S = _pair_eris(n, g)
    o = max(1, int(n * OCC_SHARE))
    if op == "fock":
        d["H"], d["P"] = _core(S, g), _densities(n, o, 1, g)[0]
    elif op == "multi":
        # response densities: symmetric, of mixed sign
        p = _densities(n, o, case["nd"] + 1, g)
        d["P"] = p[1:] - p[:1]
    elif op == "ao2mo":
        d["C"] = _orbitals(n, g)
    elif op == "mp2":
        d["C"], d["e"] = _orbitals(n, g), _energies(n, case["o"], g)
    return d


def _water(case, seed):
    return water_system(case["k"], basis="builtin:" + case["basis"], seed=seed * 1009 + case["k"], bond_jitter=0.05,
                        angle_jitter=5.0, spacing=case["spacing"])


def _batch_systems(case, seed):
    return [batch_system(s) for s in batch_specs(case["count"], seed=seed * 31 + 7)]


def prepare(case, seed):
    op = case["op"]
    st = dict(case=case)
    if op == "batch":
        b = Batch(0)
        for s in _batch_systems(case, seed):
            b.add_system(s)
        b.autotune()  # uploads the batch and picks its work-item size, once per batch
        st["batch"] = b
        return st
    ctx = st["ctx"] = hip.Context(0)
    if op == "scf":
        s = _water(case, seed)
        ctx.eri_load_packed(s.coulomb_packed(), s.nbf)
        st.update(H=s.hcore(), S=s.overlap(), VN=s.nrep(), o=s.nel // 2)
        return st
    d = _single(case, seed)
    if "m" in d:
        m = d.pop("m")
        ctx.eri_load_packed(_pack(m), case["n"])
        del m
    st.update({k: _host(v) for k, v in d.items()})
    torch.cuda.empty_cache()
    return st


# ---------------------------------------------------------------------------------------------- passes


def run(st):
    case = st["case"]
    op = case["op"]
    if op == "fock":
        return st["ctx"].fock_jk(st["H"], st["P"], case["x"])
    if op == "multi":
        return st["ctx"].fock_jk_multi(None, st["P"], case["x"])
    if op == "ao2mo":
        return st["ctx"].ao2mo(st["C"], case["o"], case["block"], "fp64")
    if op == "mp2":
        return st["ctx"].mp2(st["C"], st["e"], case["o"], case["precision"])
    if op == "eigh":
        return st["ctx"].eigh(st["A"])
    if op == "scf":
        mixed = dict(fock_precision="fp32", threshold=1e-6) if case["mixed"] else {}
        return st["ctx"].scf(st["H"], st["S"], st["VN"], st["o"], device=True, **mixed)
    return st["batch"].run()


# ---------------------------------------------------------------------------------------------- work


def _unique(n):
    p = n * (n + 1) // 2
    return p * (p + 1) // 2


def _fock_flops(n):
    return 12 * _unique(n)  # two Coulomb and four exchange products per unique integral


def _ovov_flops(n, o):
    """The four quarter transforms of (ia|jb) with ket-pair symmetry first and i >= j after it."""
    v = n - o
    return o * n * n * n * (n + 1) + o * (o + 1) * (n ** 3 + n * n * v + n * v * v)


# SCF iterations taken as the least a run does; each one reads the ERIs and forms one density.
SCF_ITERATIONS = 10


def _scf_work(n):
    return dict(bytes=SCF_ITERATIONS * 8 * _unique(n) + 56 * n * n, flops=SCF_ITERATIONS * (_fock_flops(n) + 10 * n ** 3))


def work(case):
    op = case["op"]
    if op == "batch":
        # (H2O)_k, k = 1..3, half in STO-3G (7 k) and half in cc-pVDZ (24 k); 5 k occupied
        total = dict(bytes=0.0, flops=0.0)
        for per, k in [(per, k) for per in (7, 24) for k in (1, 2, 3)]:
            w = _scf_work(per * k)
            total["bytes"] += w["bytes"] * case["count"] / 6.0
            total["flops"] += (w["flops"] + _ovov_flops(per * k, 5 * k)) * case["count"] / 6.0
        return total
    if op == "scf":
        return _scf_work(case["k"] * (24 if case["basis"] == "cc-pvdz" else 7))
    n = case["n"]
    if op == "fock":
        return dict(bytes=8 * _unique(n) + 24 * n * n, flops=_fock_flops(n))
    if op == "multi":
        return dict(bytes=8 * _unique(n) + 16 * case["nd"] * n * n, flops=case["nd"] * _fock_flops(n))
    if op == "eigh":
        return dict(bytes=16 * n * n, flops=16 * n ** 3 // 3)
    o = case["o"]
    if op == "mp2":
        return dict(bytes=8 * _unique(n) + 8 * n * n, flops=_ovov_flops(n, o))
    if case["block"] == "ovov":
        return dict(bytes=8 * _unique(n) + 8 * n * n + 8 * (o * (n - o)) ** 2, flops=_ovov_flops(n, o))
    return dict(bytes=8 * _unique(n) + 8 * n * n + 8 * n ** 4, flops=n ** 4 * (n + 1) * 4)


# ---------------------------------------------------------------------------------------------- exact values


def _pair_index(n):
    i = torch.arange(n, device="cuda")
    hi, lo = torch.maximum(i[:, None], i[None]), torch.minimum(i[:, None], i[None])
    return hi * (hi + 1) // 2 + lo


def _g_of_p(m, ij, P, x):
    """sum_rs P_rs ((pq|rs) - x (pr|qs)) for the symmetric P, from the pair matrix."""
    n = P.shape[0]
    w = torch.zeros(m.shape[0], dtype=torch.float64, device="cuda")
    w.index_add_(0, ij.reshape(-1), P.reshape(-1))
    out = (m @ w)[ij]
    step = max(1, (1 << 27) // n ** 3)
    for p in range(0, n, step):
        rows = m[ij[p:p + step]][:, :, ij]  # (p, r, q, s)
        out[p:p + step] -= x * (rows * P[None, :, None, :]).sum((1, 3))
    return out


def _transform(m, ij, C1, C3):
    """<ij|ab> = (ia|jb), i, j over the columns of C1 and a, b over those of C3."""
    n, mi, ma = C1.shape[0], C1.shape[1], C3.shape[1]
    # half-transformed bra: T[ia, pair] = sum_mu,nu C1[mu,i] C3[nu,a] (mu nu|pair)
    t = torch.zeros((mi * ma, m.shape[0]), dtype=torch.float64, device="cuda")
    for mu in range(n):
        half = C3.T @ m[ij[mu]]  # (a, pair)
        t += (C1[mu, :, None, None] * half[None]).reshape(mi * ma, -1)
    out = torch.empty((mi, mi, ma, ma), dtype=torch.float64, device="cuda")
    for i in range(mi):
        for a in range(ma):
            out[i, :, a, :] = C1.T @ t[i * ma + a][ij] @ C3
    return out


def _mp2_energy(m, ij, C, e, o):
    """Closed-shell MP2 energy, from (ia|jb) as one matrix over ia."""
    n = C.shape[0]
    v = n - o
    Co, Cv = C[:, :o], C[:, o:]
    total = 0.0
    t = torch.zeros((o * v, m.shape[0]), dtype=torch.float64, device="cuda")
    for mu in range(n):
        half = Cv.T @ m[ij[mu]]
        t += (Co[mu, :, None, None] * half[None]).reshape(o * v, -1)
    for i in range(o):
        x = t[i * v:(i + 1) * v][:, ij].reshape(v, n, n)  # (a, lam, sig)
        x = torch.matmul(torch.matmul(Co.T.contiguous(), x), Cv)  # (a, j, b)
        d = e[i] + e[:o][None, :, None] - e[o:][:, None, None] - e[o:][None, None, :]
        total += float((x * (2.0 * x - x.transpose(0, 2)) / d).sum())
    return total


def _scf_exact(H, S, VN, o, m):
    """RHF to far below the passes' threshold: DIIS on the dense matrices."""
    n = H.shape[0]
    ij = _pair_index(n)
    H, S = torch.from_numpy(H).cuda(), torch.from_numpy(S).cuda()
    w, u = np.linalg.eigh(_host(S))
    X = torch.from_numpy((u / np.sqrt(w)) @ u.T).cuda()

    def levels(F):
        e, c = np.linalg.eigh(_host(X @ F @ X))
        return torch.from_numpy(e).cuda(), X @ torch.from_numpy(c).cuda()

    C = levels(H)[1]
    P = 2.0 * C[:, :o] @ C[:, :o].T
    fs, es, last = [], [], None
    for _ in range(80):
        F = H + _g_of_p(m, ij, P, 0.5)
        E = 0.5 * float((P * (H + F)).sum()) + VN
        r = X @ (F @ P @ S - S @ P @ F) @ X
        if float(r.abs().max()) < 1e-11 or (last is not None and float(r.abs().max()) < 1e-9 and abs(E - last) < 1e-12):
            break
        last = E
        fs, es = (fs + [F])[-8:], (es + [r])[-8:]
        k = len(fs)
        B = np.full((k + 1, k + 1), -1.0)
        B[k, k] = 0.0
        B[:k, :k] = [[float((a * b).sum()) for b in es] for a in es]
        B[:k, :k] /= max(B[k - 1, k - 1], 1e-300)
        c = np.linalg.lstsq(B, np.append(np.zeros(k), -1.0), rcond=None)[0][:k]
        F = sum(float(x) * f for x, f in zip(c, fs))
        e, C = levels(F)
        P = 2.0 * C[:, :o] @ C[:, :o].T
    e, C = levels(F)
    return E, e, C, P, F


def _pairs_of(packed, n):
    p = n * (n + 1) // 2
    m = torch.zeros((p, p), dtype=torch.float64, device="cuda")
    m[torch.ones((p, p), dtype=torch.bool, device="cuda").tril_()] = torch.from_numpy(packed).cuda()
    return m + torch.tril(m, -1).T


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        E, Ec = [], []
        for s in _batch_systems(case, seed):
            o, m = s.nel // 2, _pairs_of(s.coulomb_packed(), s.nbf)
            en, e, C, _, _ = _scf_exact(s.hcore(), s.overlap(), s.nrep(), o, m)
            E.append(en)
            Ec.append(_mp2_energy(m, _pair_index(s.nbf), C, e, o))
        return dict(E_rhf=np.array(E), E_corr=np.array(Ec), iterations=None, status=None)
    if op == "scf":
        s = _water(case, seed)
        m = _pairs_of(s.coulomb_packed(), s.nbf)
        E, e, _, P, F = _scf_exact(s.hcore(), s.overlap(), s.nrep(), s.nel // 2, m)
        return dict(E=E, iterations=None, C=None, e=_host(e), P=_host(P), F=_host(F))  # C: signs are free
    d = _single(case, seed)
    if op == "eigh":
        return np.linalg.eigvalsh(_host(d["A"])), None  # eigenvectors: signs are free
    n = case["n"]
    ij = _pair_index(n)
    if op == "fock":
        return _host(d["H"] + _g_of_p(d["m"], ij, d["P"], case["x"]))
    if op == "multi":
        return _host(torch.stack([_g_of_p(d["m"], ij, p, case["x"]) for p in d["P"]]))
    if op == "ao2mo":
        o, C = case["o"], d["C"]
        return _host(_transform(d["m"], ij, C, C) if case["block"] == "full" else _transform(d["m"], ij, C[:, :o], C[:, o:]))
    return _mp2_energy(d["m"], ij, d["C"], d["e"], case["o"])
