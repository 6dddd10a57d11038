"""Timed workloads of the GW engine: what its users have it compute.

Each case goes through a public entry point (quack_amd.gw, quack_amd.scf) the
way a program calls it; the kinds are

  oneshot  QuAcK's RG0W0 call on host MO integrals (handle made and dropped)
  g0w0     a kept engine, AO integrals in HBM: AO->MO block, then G0W0
  evgw     the same, then evGW to self-consistency (DIIS 5)
  lattice  evGW of a hydrogen lattice with its own integrals and RHF
  batch    a group of equal molecules: AO->MO, then batched G0W0 or evGW
  df       density-fitted screening and one self-energy sweep
  ug0w0    QuAcK's UG0W0 call on host MO integrals of two spins
  phbse    QuAcK's RGW_phBSE call (singlets and triplets) on host integrals
  jk       one Fock build over AO integrals in HBM

Integrals other than the lattice's are synthetic density-fitted Gram
matrices, (pq|rs) = sum_P B_P,pq B_P,rs with B_P,pq decaying in |p - q| and
energies spread as a hydrogen chain's: 8-fold symmetric, positive definite and
cheap to make at any size.
"""
import math

import numpy as np
import torch

from quack_amd import gw, scf
from quack_amd import intgen, workloads


def listed():
    return [
        # water in cc-pVDZ through the drop-in call: launches and latency
        {"name": "oneshot-n24", "kind": "oneshot", "N": 24, "nO": 5, "method": "graph"},
        # the H10 chain's size (N = 50, 225 pairs) with QuAcK's SRG option
        {"name": "g0w0-n50-srg", "kind": "g0w0", "N": 50, "nO": 5, "method": "srg"},
        # an ordinary molecule, odd sizes, linearised QP, own full solves
        {"name": "g0w0-n115-sytrd", "kind": "g0w0", "N": 115, "nO": 13, "method": "linear", "eig": "sytrd"},
        # the 5 x 6 lattice's size (2025 pairs), every default
        {"name": "g0w0-n150", "kind": "g0w0", "N": 150, "nO": 15, "method": "graph", "eig": "syevd"},
        # evGW in plain FP64, every default
        {"name": "evgw-n100", "kind": "evgw", "N": 100, "nO": 10, "eig": "syevd"},
        # the headline molecule: H50 lattice, split precision, refined solves
        {"name": "lattice-5x10", "kind": "lattice", "nx": 5, "ny": 10, "precision": "mixed2",
         "eig": "refine+sytrd", "de_max": 0.01},
        # batches of small molecules: G0W0 in FP64, evGW in split precision with replayed cycles
        {"name": "batch-g0w0-24xn60", "kind": "batch", "nmol": 24, "N": 60, "nO": 6, "method": "g0w0",
         "precision": "fp64"},
        {"name": "batch-evgw-8xn90", "kind": "batch", "nmol": 8, "N": 90, "nO": 9, "method": "evgw",
         "precision": "mixed2"},
        # density-fitted precision form at half the 600-orbital workload's size
        {"name": "df-n300", "kind": "df", "N": 300, "nO": 30, "naux": 900, "precision": "mixed"},
        # open shell: the H10 chain's size with one electron removed
        {"name": "ug0w0-n50", "kind": "ug0w0", "N": 50, "nOa": 6, "nOb": 5},
        # Bethe-Salpeter on top of a G0W0
        {"name": "phbse-n60", "kind": "phbse", "N": 60, "nO": 6},
        # a Fock build of a 200-function molecule, once per SCF cycle
        {"name": "jk-n200", "kind": "jk", "N": 200, "nO": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["oneshot", "g0w0", "evgw", "lattice", "batch", "df", "ug0w0", "phbse", "jk"])
    if kind == "oneshot":
        N = _log(rng, 10, 60)
        return {"kind": kind, "N": N, "nO": rng.randint(1, max(1, N // 4)), "method": rng.choice(["graph", "linear", "srg"])}
    if kind == "g0w0":
        N = _log(rng, 30, 170)
        return {"kind": kind, "N": N, "nO": max(1, N // rng.randint(8, 12)), "method": rng.choice(["graph", "linear", "srg"]),
                "eig": rng.choice(["syevd", "sytrd"])}
    if kind == "evgw":
        N = _log(rng, 30, 130)
        return {"kind": kind, "N": N, "nO": max(1, N // rng.randint(8, 12)),
                "eig": rng.choice(["syevd", "sytrd", "refine+sytrd"])}
    if kind == "lattice":
        nx, ny = rng.choice([(2, 5), (2, 7), (3, 4), (2, 9), (4, 5), (4, 6), (4, 7), (5, 6), (4, 9), (5, 8)])
        return {"kind": kind, "nx": nx, "ny": ny, "precision": rng.choice(["fp64", "mixed2"]),
                "eig": "refine+sytrd", "de_max": 0.01}
    if kind == "batch":
        N = _log(rng, 20, 120)
        method = rng.choice(["g0w0", "evgw"])
        return {"kind": kind, "nmol": rng.randint(2, max(3, (1500 if method == "g0w0" else 700) // N)), "N": N,
                "nO": max(1, N // 10), "method": method, "precision": rng.choice(["fp64", "mixed2"])}
    if kind == "df":
        N = _log(rng, 60, 300)
        return {"kind": kind, "N": N, "nO": max(2, N // 10), "naux": 3 * N + rng.randint(-5, 5),
                "precision": rng.choice(["fp64", "mixed", "mixed2"])}
    if kind == "ug0w0":
        N = _log(rng, 16, 70)
        nOb = max(1, N // 10)
        return {"kind": kind, "N": N, "nOa": nOb + rng.randint(0, 2), "nOb": nOb}
    if kind == "phbse":
        N = _log(rng, 20, 80)
        return {"kind": kind, "N": N, "nO": max(2, N // 10)}
    N = _log(rng, 50, 240)
    return {"kind": kind, "N": N, "nO": max(1, N // 10)}


# ---- inputs -----------------------------------------------------------------

def _energies(rng, N, nO):
    return np.concatenate([np.sort(rng.uniform(-1.1, -0.35, nO)), np.sort(rng.uniform(0.15, 4.0, N - nO))])


def _factors(rng, N, nO, naux=None, kmax=0.2):
    """(e, B[P, p, q]) with the largest (ia|ia) equal to kmax."""
    e = _energies(rng, N, nO)
    G = rng.standard_normal((naux or 2 * N, N, N))
    B = np.triu(G) + np.transpose(np.triu(G, 1), (0, 2, 1))
    p = np.arange(N)
    B *= np.exp(-np.abs(p[:, None] - p[None, :]) / (N / 6.0))
    ov = B[:, :nO, nO:]
    return e, B * math.sqrt(kmax / np.einsum("Pia,Pia->ia", ov, ov).max())


def _orbitals(rng, N):
    """Orthogonal MO coefficients, mixing neighbouring functions as localised orbitals do."""
    A = rng.standard_normal((N, N))
    p = np.arange(N)
    A = (A - A.T) * 0.2 * np.exp(-np.abs(p[:, None] - p[None, :]) / 4.0)
    return np.linalg.solve(np.eye(N) + A, np.eye(N) - A)  # Cayley transform


def _ao_eri(B, c):
    """Device AO integrals <mu nu|la si> (mu fastest) whose MO factors are B: AO factors c B c^T."""
    N = c.shape[0]
    ct = torch.from_numpy(c).cuda()
    A = (ct @ torch.from_numpy(B).cuda() @ ct.T.contiguous()).reshape(B.shape[0], N * N)
    chem = (A.T.contiguous() @ A).view(N, N, N, N)           # (mu la|nu si)
    return chem.permute(3, 1, 2, 0).contiguous().view(-1)    # [si, la, nu, mu]


def _mo_eri(Bl, Br):
    """Host <pq|rs> (p fastest) = sum_P Bl[P, p, r] Br[P, q, s]."""
    N, Q = Bl.shape[1], Br.shape[1]
    chem = (Bl.reshape(Bl.shape[0], -1).T @ Br.reshape(Br.shape[0], -1)).reshape(N, N, Q, Q)  # [p, r, q, s]
    return np.ascontiguousarray(chem.transpose(3, 1, 2, 0)).reshape(-1)


def _options(method):
    return {"graph": {"eta": 0.1}, "linear": {"eta": 0.05, "linearize": True}, "srg": {"doSRG": True}}[method]


def _host_inputs(case, seed):
    """The inputs made on the host: what prepare() hands over and exact() starts from."""
    rng = np.random.default_rng([seed, 20])
    kind = case["kind"]
    if kind == "batch":
        mols = []
        for _ in range(case["nmol"]):
            e, B = _factors(rng, case["N"], case["nO"])
            mols.append((e, B, _orbitals(rng, case["N"])))
        return mols
    if kind == "ug0w0":
        N = case["N"]
        ea, Ba = _factors(rng, N, case["nOa"])
        U = _orbitals(rng, N)  # beta orbitals: a rotation of the alpha ones
        U = np.linalg.solve(np.eye(N) * 3.0 + U, np.eye(N) * 3.0 + U.T)
        Bb = np.matmul(np.matmul(U.T, Ba), U)
        eb = np.concatenate([np.sort(rng.uniform(-1.1, -0.35, case["nOb"])),
                             np.sort(rng.uniform(0.15, 4.0, N - case["nOb"]))])
        return np.stack([ea, eb], axis=1), Ba, Bb
    if kind == "jk":
        e, B = _factors(rng, case["N"], case["nO"])
        c = _orbitals(rng, case["N"])
        return B, c, 2.0 * c[:, :case["nO"]] @ c[:, :case["nO"]].T
    e, B = _factors(rng, case["N"], case["nO"])
    if kind == "phbse":
        shift = 0.05 * rng.standard_normal(case["N"]) + np.where(np.arange(case["N"]) < case["nO"], -0.1, 0.1)
        return e, e + shift, B
    return e, B, _orbitals(rng, case["N"])


def _lattice(case, seed):
    for k in range(8):  # a geometry whose RHF does not converge is replaced
        mol = intgen.h_lattice(case["nx"], case["ny"], seed=seed + 1000003 * k)
        try:
            return mol, workloads.device_inputs(mol)
        except RuntimeError as ex:
            if isinstance(ex, gw.QKError):
                raise
    raise RuntimeError("no converged RHF")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "lattice":
        mol, (hf, eri, c) = _lattice(case, seed)
        g = gw.GWEngine(mol.nBas, hf["nOrb"], mol.nO)
        g.set_precision(case["precision"])
        g.set_eigensolver(case["eig"], case["de_max"])
        return {"case": case, "g": g, "eri": eri, "c": c, "e": hf["eHF"]}
    if kind == "df":
        N, nO, naux = case["N"], case["nO"], case["naux"]
        gen = torch.Generator("cuda").manual_seed(seed + 7)
        G = torch.randn((N, N, naux), generator=gen, device="cuda", dtype=torch.float64)  # [q, p, P]
        p = torch.arange(N, device="cuda", dtype=torch.float64)
        G = torch.where((p[:, None] <= p[None, :])[:, :, None], G, G.transpose(0, 1))
        G = G * torch.exp(-(p[:, None] - p[None, :]).abs() / (N / 6.0))[:, :, None]
        ov = G[nO:, :nO]
        B = (G * torch.sqrt(0.2 / (ov * ov).sum(dim=2).max())).contiguous()
        rng = np.random.default_rng([seed, 21])
        e = _energies(rng, N, nO)
        g = gw.GWEngine(N, N, nO)
        g.set_precision(case["precision"])
        g.set_eigensolver("sytrd")
        torch.cuda.synchronize()
        g.set_eri_df_device(B.data_ptr(), naux)
        return {"case": case, "g": g, "e": e, "w": e + 0.05 * rng.standard_normal(N)}
    x = _host_inputs(case, seed)
    if kind == "oneshot":
        e, B, _ = x
        return {"case": case, "e": e, "eri": _mo_eri(B, B)}
    if kind == "ug0w0":
        e, Ba, Bb = x
        return {"case": case, "e": e, "aa": _mo_eri(Ba, Ba), "ab": _mo_eri(Ba, Bb), "bb": _mo_eri(Bb, Bb)}
    if kind == "phbse":
        eW, eGW, B = x
        return {"case": case, "eW": eW, "eGW": eGW, "eri": _mo_eri(B, B)}
    if kind == "jk":
        B, c, P = x
        eri = _ao_eri(B, c)
        torch.cuda.synchronize()
        return {"case": case, "jk": scf.JK(case["N"]), "eri": eri, "P": P}
    if kind == "batch":
        eri = torch.stack([_ao_eri(B, c) for _, B, c in x])
        cc = torch.stack([torch.from_numpy(np.ascontiguousarray(c.T)).view(-1) for _, _, c in x]).cuda()
        b = gw.GWBatch(case["nmol"], case["N"], case["N"], case["nO"])
        b.set_precision(case["precision"])
        b.set_graphs(True)
        torch.cuda.synchronize()
        return {"case": case, "b": b, "eri": eri, "c": cc, "e": np.stack([e for e, _, _ in x])}
    e, B, c = x
    eri = _ao_eri(B, c)
    ct = torch.from_numpy(np.ascontiguousarray(c.T)).view(-1).cuda()  # column-major
    g = gw.GWEngine(case["N"], case["N"], case["nO"])
    if "eig" in case:
        g.set_eigensolver(case["eig"])
    torch.cuda.synchronize()
    return {"case": case, "g": g, "eri": eri, "c": ct, "e": e}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "oneshot":
        return gw.RG0W0(state["eri"], state["e"], case["nO"], **_options(case["method"]))
    if kind == "g0w0":
        g = state["g"]
        g.set_eri_ao_device(state["eri"].data_ptr(), state["c"].data_ptr())
        return g.g0w0(state["e"], **_options(case["method"]))
    if kind in ("evgw", "lattice"):
        g = state["g"]
        g.set_eri_ao_device(state["eri"].data_ptr(), state["c"].data_ptr())
        return g.evgw(state["e"], thresh=1e-6, max_diis=5, eta=0.1)
    if kind == "batch":
        b, eri, c = state["b"], state["eri"], state["c"]
        b.set_eri_ao_device(eri.data_ptr(), eri.shape[1], c.data_ptr(), c.shape[1])
        if case["method"] == "evgw":
            return b.evgw(state["e"], thresh=1e-6, max_diis=5, eta=0.1)
        return b.g0w0(state["e"], doSRG=True)
    if kind == "df":
        g = state["g"]
        g.screen(state["e"])
        return g.sigma_at(state["e"], state["w"], eta=0.1)
    if kind == "ug0w0":
        return gw.UG0W0(state["aa"], state["ab"], state["bb"], state["e"], (case["nOa"], case["nOb"]), eta=0.1)
    if kind == "phbse":
        r = gw.RGW_phBSE(state["eri"], state["eW"], state["eGW"], case["nO"], eta=0.05)
        return {k: r[k] for k in ("EcBSE", "OmS", "OmT")}
    return state["jk"](state["eri"].data_ptr(), state["P"])


# ---- work -------------------------------------------------------------------

def _aotomo_flops(N, nO):
    v = N - nO
    return 2.0 * N ** 4 * nO + 2.0 * N ** 3 * v * nO + 4.0 * N ** 3 * v * nO


def _eig_flops(S, vectors):
    """Tridiagonalisation (4/3 S^3); with vectors, their back-transformation (2 S^3) and a
    divide and conquer on the tridiagonal (4/3 S^3)."""
    return (4.0 / 3.0 + (10.0 / 3.0 if vectors else 0.0)) * S ** 3


def work(case):
    kind = case["kind"]
    if kind == "lattice":
        atoms = case["nx"] * case["ny"]
        N, nO = 5 * atoms, atoms // 2
        S = nO * (N - nO)
        # six cycles: 3 full solves, the others as one solve's refinement
        return {"bytes": 8.0 * N ** 4, "flops": _aotomo_flops(N, nO) + 6 * (_eig_flops(S, True) + 2.0 * N * N * S * S)}
    N = case["N"]
    if kind == "jk":
        return {"bytes": 8.0 * (N ** 4 + 3 * N * N), "flops": 4.0 * N ** 4}
    if kind == "ug0w0":
        S = case["nOa"] * (N - case["nOa"]) + case["nOb"] * (N - case["nOb"])
        return {"bytes": 8.0 * 3 * N ** 4, "flops": _eig_flops(S, True) + _eig_flops(S, False) + 4.0 * N * N * S * S}
    S = case["nO"] * (N - case["nO"])
    full = _eig_flops(S, True) + 2.0 * N * N * S * S
    if kind == "oneshot":
        return {"bytes": 8.0 * (N * N * S + N * N), "flops": full + _eig_flops(S, False)}
    if kind == "phbse":
        # screening, then singlet and triplet problems with two eigensolves and four products each
        return {"bytes": 8.0 * N ** 4, "flops": full + 2 * (2 * _eig_flops(S, True) + 8.0 * S ** 3) + 4.0 * S ** 3}
    if kind == "df":
        x = case["naux"]
        return {"bytes": 8.0 * x * N * N, "flops": _eig_flops(S, True) + 2.0 * x * S * S + 2.0 * x * N * N * S}
    if kind == "batch":
        one = 5 * full if case["method"] == "evgw" else full + _eig_flops(S, False)
        return {"bytes": 8.0 * case["nmol"] * N ** 4, "flops": case["nmol"] * (_aotomo_flops(N, case["nO"]) + one)}
    one = 5 * full if kind == "evgw" else full + _eig_flops(S, False)
    return {"bytes": 8.0 * N ** 4, "flops": _aotomo_flops(N, case["nO"]) + one}


# ---- 64-bit values in numpy -------------------------------------------------

def _rpa(d, Kia, f, vectors=True):
    """dRPA of pair energies d and coupling (ia|jb): A - B = diag(d), A + B = diag(d) + f K."""
    sd = np.sqrt(d)
    C = f * (sd[:, None] * Kia * sd[None, :])
    C[np.diag_indices(len(d))] += d * d
    if not vectors:
        Om = np.sqrt(np.linalg.eigvalsh(C))
        return 0.5 * (Om.sum() - (d + 0.5 * f * np.diag(Kia)).sum())
    w, Z = np.linalg.eigh(C)
    Om = np.sqrt(w)
    W = Z * (sd[:, None] / np.sqrt(Om)[None, :])
    return 0.5 * (Om.sum() - (d + 0.5 * f * np.diag(Kia)).sum()), Om, W


def _weights(w, e, Om, r2, nO, eta, srg):
    """Sig and dSig of every orbital at w from r2[p, q, m] = 2 rho^2, poles at e_q -+ Om_m."""
    sig, dsig = np.zeros(len(e)), np.zeros(len(e))
    for q in range(len(e)):
        x = w[:, None] - e[q] + (Om if q < nO else -Om)[None, :]
        x2 = x * x
        if srg:
            t = r2[:, q] * (1.0 - np.exp(-1000.0 * x2)) / x
            sig += t.sum(axis=1)
            dsig -= (t / x).sum(axis=1)
        else:
            t = r2[:, q] / (x2 + eta * eta)
            sig += (t * x).sum(axis=1)
            dsig -= (t * (x2 - eta * eta) / (x2 + eta * eta)).sum(axis=1)
    return sig, dsig


def _galitskii_migdal(e, Om, r2, nO, eta, srg):
    x = e[nO:, None, None] - e[None, :nO, None] + Om[None, None, :]
    t = r2[nO:, :nO] * 2.0
    return -float((t * (1.0 - np.exp(-1000.0 * x * x)) / x).sum() if srg else (t * x / (x * x + eta * eta)).sum())


def _newton(e0, eG, Om, r2, nO, start, Z, eta, srg):
    w, Z, live = start.copy(), Z.copy(), np.ones(len(e0), bool)
    for it in range(1, 65):
        p = np.flatnonzero(live)
        s, ds = _weights(w[p], eG, Om, r2[p], nO, eta, srg) if len(p) == len(e0) else _rows(w, p, eG, Om, r2, nO, eta, srg)
        f, df = w[p] - e0[p] - s, 1.0 / (1.0 - ds)
        w[p] -= df * f
        stop = ~(np.abs(f) > 1e-6)
        if it == 64:
            w[p] = start[p]
            break
        Z[p[stop]] = df[stop]
        live[p[stop]] = False
        if not live.any():
            break
    return w, Z


def _rows(w, p, e, Om, r2, nO, eta, srg):
    sig, dsig = np.zeros(len(p)), np.zeros(len(p))
    for k, i in enumerate(p):
        x = w[i] - e[:, None] + np.where(np.arange(len(e)) < nO, 1.0, -1.0)[:, None] * Om[None, :]
        x2 = x * x
        if srg:
            t = r2[i] * (1.0 - np.exp(-1000.0 * x2)) / x
            sig[k], dsig[k] = t.sum(), -(t / x).sum()
        else:
            t = r2[i] / (x2 + eta * eta)
            sig[k], dsig[k] = (t * x).sum(), -(t * (x2 - eta * eta) / (x2 + eta * eta)).sum()
    return sig, dsig


def _pairs(e, nO):
    return (e[None, nO:] - e[:nO, None]).reshape(-1)


def _density2(B, T):
    """2 rho(p, q, m)^2 with rho = sum_P B[P, p, q] T[P, m]."""
    n = B.shape[1]
    r = (B.reshape(B.shape[0], -1).T @ T).reshape(n, n, -1)
    return 2.0 * r * r


def _sigma(e, Om, r2, nO, eta, srg):
    s, ds = _weights(e, e, Om, r2, nO, eta, srg)
    return s, 1.0 / (1.0 - ds), _galitskii_migdal(e, Om, r2, nO, eta, srg)


def _g0w0(e, B, nO, eta=0.0, linearize=False, doSRG=False):
    Bov = B[:, :nO, nO:].reshape(B.shape[0], -1)
    K = Bov.T @ Bov
    _, Om, W = _rpa(_pairs(e, nO), K, 4.0)
    r2 = _density2(B, Bov @ W)
    Sig, Z, Egm = _sigma(e, Om, r2, nO, eta, doSRG)
    lin = e + Z * Sig
    eGW = lin
    if not linearize:
        eGW, Z = _newton(e, e, Om, r2, nO, lin, Z, eta, doSRG)
    return {"eGW": eGW, "SigC": Sig, "Z": Z, "Om": Om, "EcRPA": _rpa(_pairs(eGW, nO), K, 4.0, False), "EcGM": Egm}


def _evgw(e0, B, nO, eta=0.1, thresh=1e-6, max_diis=5):
    Bov = B[:, :nO, nO:].reshape(B.shape[0], -1)
    K = Bov.T @ Bov
    e, Z, errs, vals, cycles, conv = e0.copy(), np.ones(len(e0)), [], [], 0, 1.0
    while conv > thresh and cycles <= 256:
        Ec, Om, W = _rpa(_pairs(e, nO), K, 4.0)
        r2 = _density2(B, Bov @ W)
        Sig, Z, Egm = _sigma(e, Om, r2, nO, eta, False)
        new, Z = _newton(e0, e, Om, r2, nO, e, Z, eta, False)
        conv = np.abs(new - e).max()
        errs, vals = [new - e] + errs[:max_diis - 1], [new] + vals[:max_diis - 1]
        m = len(errs)
        A = -np.ones((m + 1, m + 1))
        A[m, m] = 0.0
        A[:m, :m] = np.array(errs) @ np.array(errs).T
        if 1.0 / np.linalg.cond(A, 1) > 1e-13:
            x = np.linalg.solve(A, np.concatenate([np.zeros(m), [-1.0]]))
            new = np.array(vals).T @ x[:m]
        e = new
        cycles += 1
    return {"eGW": e, "SigC": Sig, "Z": Z, "Om": Om, "EcRPA": Ec, "EcGM": Egm, "nSCF": cycles}


def _ug0w0(e, Ba, Bb, nO, eta):
    B = (Ba, Bb)
    ov = np.concatenate([B[s][:, :nO[s], nO[s]:].reshape(Ba.shape[0], -1) for s in range(2)], axis=1)
    pairs = lambda x: np.concatenate([_pairs(x[:, s], nO[s]) for s in range(2)])
    K = ov.T @ ov
    _, Om, W = _rpa(pairs(e), K, 2.0)
    T = ov @ W
    eGW, Sig, Z, Egm = np.zeros_like(e), np.zeros_like(e), np.zeros_like(e), np.zeros(2)
    for s in range(2):
        r2 = _density2(B[s], T) * 0.5
        Sig[:, s], z, ec = _sigma(e[:, s], Om, r2, nO[s], eta, False)
        Egm[s] = 0.5 * ec
        eGW[:, s], Z[:, s] = _newton(e[:, s], e[:, s], Om, r2, nO[s], e[:, s] + z * Sig[:, s], z, eta, False)
    return {"eGW": eGW, "SigC": Sig, "Z": Z, "Om": Om, "EcRPA": _rpa(pairs(eGW), K, 2.0, False), "EcGM": Egm}


def _phbse(eW, eGW, B, nO, eta):
    n, v = len(eW), len(eW) - nO
    S = nO * v
    Bov = B[:, :nO, nO:].reshape(B.shape[0], -1)
    K = Bov.T @ Bov
    _, Om, W = _rpa(_pairs(eW, nO), K, 4.0)
    T = Bov @ W
    U = T * (4.0 * Om / (Om ** 2 + eta ** 2))[None, :] @ T.T  # 4 sum_m w_m T T^T between factors
    Boo, Bvv, Bia = B[:, :nO, :nO], B[:, nO:, nO:], B[:, :nO, nO:]
    UB = np.tensordot(U, Bvv, axes=(1, 0))
    UBia = np.tensordot(U, Bia, axes=(1, 0))
    KA = np.tensordot(Boo, UB - Bvv, axes=(0, 0)).transpose(0, 2, 1, 3).reshape(S, S)      # [i j a b] -> ia, jb
    KB = np.tensordot(Bia, UBia - Bia, axes=(0, 0)).transpose(0, 3, 2, 1).reshape(S, S)    # [i b j a] -> ia, jb
    Ec, Oms = [], []
    for f in (2.0, 0.0):
        A, Bm = np.diag(_pairs(eGW, nO)) + f * K + KA, f * K + KB
        x, Q = np.linalg.eigh(A - Bm)
        R = (Q * np.sqrt(x)) @ Q.T
        M = R @ (A + Bm) @ R
        O = np.sqrt(np.linalg.eigvalsh(0.5 * (M + M.T)))
        Ec.append(0.5 * (O.sum() - np.trace(A)))
        Oms.append(O)
    return {"EcBSE": np.array([Ec[0], 3.0 * Ec[1]]), "OmS": Oms[0], "OmT": Oms[1]}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("lattice", "df") or (kind != "jk" and case["N"] > 150) or (kind == "evgw" and case["N"] > 110):
        return None  # minutes of LAPACK
    if kind == "batch" and case["nmol"] * case["N"] ** 5 * (5 if case["method"] == "evgw" else 1) > 3e11:
        return None
    x = _host_inputs(case, seed)
    if kind in ("oneshot", "g0w0"):
        e, B, _ = x
        return _g0w0(e, B, case["nO"], **_options(case["method"]))
    if kind == "evgw":
        e, B, _ = x
        return _evgw(e, B, case["nO"])
    if kind == "batch":
        r = [_evgw(e, B, case["nO"]) if case["method"] == "evgw" else _g0w0(e, B, case["nO"], doSRG=True)
             for e, B, _ in x]
        return {k: np.array([m[k] for m in r]) for k in r[0]}
    if kind == "ug0w0":
        e, Ba, Bb = x
        return _ug0w0(e, Ba, Bb, (case["nOa"], case["nOb"]), 0.1)
    if kind == "phbse":
        eW, eGW, B = x
        return _phbse(eW, eGW, B, case["nO"], 0.05)
    B, c, P = x
    A = np.matmul(np.matmul(c, B), c.T)
    J = np.tensordot(np.tensordot(A, P, axes=([1, 2], [0, 1])), A, axes=(0, 0))
    AP = np.matmul(A, P)
    return J, -np.tensordot(AP, A, axes=([0, 2], [0, 2]))
