"""GPU: the full RPA eigensolve at the sizes where its kernels change shape,
against LAPACK (numpy) on the same matrix.

The number of pairs nS = nO nV is the order of the matrix; the sizes sit on
both sides of every register layout of the tridiagonalisation and include
orders of one, two and odd or prime ones.  Tolerances: the matrix is built with
some 20 roundings an element (a 12-term sum, three products, the diagonal) on
either side, and the eigenvalues of either backward-stable solve are off by at
most n eps max|lambda|, so lambda differs by (2 n + 40) eps lambda_max and
Om = sqrt(lambda) by that over 2 Om, and one rounding; EcRPA is half a sum of n
such values; the self-energy is a sum over all modes, insensitive to rotations
of close ones, held to 1e-10 of its largest value.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def system(nO, nV, seed):
    rng = np.random.default_rng(seed)
    n, naux = nO + nV, 12
    e = np.concatenate([np.sort(rng.uniform(-1.5, -0.3, nO)), np.sort(rng.uniform(0.1, 4.0, nV))])
    B = 0.02 * rng.standard_normal((naux, n, n))
    return e, B + B.transpose(0, 2, 1)


def reference(e, B, nO, sigma):
    n = len(e)
    Bov = B[:, :nO, nO:].reshape(len(B), -1)
    d = (e[None, nO:] - e[:nO, None]).reshape(-1)
    sd = np.sqrt(d)
    C = 4.0 * (Bov * sd).T @ (Bov * sd)
    trace = d.sum() + 2.0 * (Bov * Bov).sum()
    C[np.diag_indices(len(d))] += d * d
    lam, Z = np.linalg.eigh(C) if sigma else (np.linalg.eigvalsh(C), None)
    Om = np.sqrt(lam)
    out = {"Om": Om, "EcRPA": 0.5 * (Om.sum() - trace), "lmax": lam[-1]}
    if sigma:
        T = Bov @ (Z * (sd[:, None] / np.sqrt(Om)[None, :]))
        rho2 = 2.0 * (B.reshape(len(B), -1).T @ T).reshape(n, n, -1) ** 2
        sgn = np.where(np.arange(n) < nO, 1.0, -1.0)
        x = e[:, None, None] - e[None, :, None] + sgn[None, :, None] * Om[None, None, :]
        out["SigC"] = (rho2 * x / (x * x + 0.01)).sum(axis=(1, 2))
    return out


def om_tolerance(ref):
    n = len(ref["Om"])
    return (2 * n + 40) * EPS * ref["lmax"] / (2.0 * ref["Om"]) + EPS * ref["Om"]


# (nO, nV): orders 1, 2, 5, 63, 64, 65, 128, 129, 160, 161, 192, 193, 256, 257, 384, 385, 512, 513,
# 1024, 1025, 1536, 1537, 2048, 2050, 2560, 2561, 3072, 3073
SHAPES = [(1, 1), (1, 2), (1, 5), (7, 9), (4, 16), (5, 13), (8, 16), (3, 43), (8, 20), (7, 23), (8, 24), (1, 193),
          (8, 32), (1, 257), (12, 32), (11, 35), (16, 32), (19, 27), (16, 64), (25, 41), (24, 64), (29, 53), (32, 64),
          (41, 50), (40, 64), (13, 197), (48, 64), (7, 439)]


@pytest.mark.parametrize("nO,nV", SHAPES)
def test_full_solve_edges(nO, nV):
    from quack_amd import gw
    nS = nO * nV
    print("full solve nS", nS, flush=True)
    e, B = system(nO, nV, nS)
    ref = reference(e, B, nO, nS <= 600)
    tol = om_tolerance(ref)
    for mode in ("sytrd", "syevd"):
        with gw.GWEngine(nO + nV, nO + nV, nO) as g:
            g.set_eri_df(B)
            g.set_eigensolver(mode)
            g.screen(e)
            sig, _ = g.sigma_at(e, e, eta=0.1)
            r = g.g0w0(e, eta=0.1, linearize=True)
        assert (np.abs(r["Om"] - ref["Om"]) <= tol).all(), mode
        if "SigC" in ref:
            for s in (sig, r["SigC"]):
                assert np.abs(s - ref["SigC"]).max() <= 1e-10 * np.abs(ref["SigC"]).max(), mode
        # the values-only solve at the quasiparticle energies
        ref2 = reference(r["eGW"], B, nO, False)
        tol2 = 0.5 * om_tolerance(ref2).sum() + nS * EPS * ref2["Om"].sum()
        assert abs(r["EcRPA"] - ref2["EcRPA"]) <= tol2, mode
    sys.stdout.flush()


@pytest.mark.parametrize("coupling", [0.0, 1e-9, 1e-5, 1e-3])
def test_full_solve_equal_poles(coupling):
    """Evenly spaced orbital energies: most pair energies coincide, so that the divide and
    conquer deflates nearly everything (coupling 0), rotates close poles, or
    solves for roots next to their poles."""
    from quack_amd import gw
    print("full solve, equal poles, coupling", coupling, flush=True)
    nO, nV = 9, 33
    e, B = system(nO, nV, 3)
    e = np.concatenate([-1.0 + 0.05 * np.arange(nO), 0.2 + 0.05 * np.arange(nV)])
    B = B * (coupling / 0.02)
    ref = reference(e, B, nO, True)
    for mode in ("sytrd", "syevd"):
        with gw.GWEngine(nO + nV, nO + nV, nO) as g:
            g.set_eri_df(B)
            g.set_eigensolver(mode)
            g.screen(e)
            sig, _ = g.sigma_at(e, e, eta=0.1)
            r = g.g0w0(e, eta=0.1, linearize=True)
        assert (np.abs(r["Om"] - ref["Om"]) <= om_tolerance(ref)).all(), mode
        for s in (sig, r["SigC"]):
            assert np.abs(s - ref["SigC"]).max() <= 1e-10 * np.abs(ref["SigC"]).max(), mode


@pytest.mark.parametrize("nmol", [3, 40, 60])
def test_batched_full_solve(nmol):
    """nS = 171 a molecule: every workgroup a CU of its own (3), fewer workgroups a
    matrix (40), more matrices than one launch holds (60)."""
    from quack_amd import gw
    print("batched full solve", nmol, flush=True)
    nO, nV = 9, 19
    n = nO + nV
    sys_ = [system(nO, nV, 100 + m) for m in range(nmol)]
    with gw.GWBatch(nmol, n, n, nO) as b:
        for m, (_, B) in enumerate(sys_):
            chem = np.einsum("Ppq,Prs->pqrs", B, B, optimize=True)
            b.set_eri_mo(m, np.asfortranarray(chem.transpose(0, 2, 1, 3)))
        r = b.g0w0(np.stack([e for e, _ in sys_]), eta=0.1, linearize=True)
    for m, (e, B) in enumerate(sys_):
        ref = reference(e, B, nO, True)
        assert (np.abs(r["Om"][m] - ref["Om"]) <= om_tolerance(ref)).all(), m
        assert np.abs(r["SigC"][m] - ref["SigC"]).max() <= 1e-10 * np.abs(ref["SigC"]).max(), m
        ref2 = reference(r["eGW"][m], B, nO, False)
        tol2 = 0.5 * om_tolerance(ref2).sum() + n * n * EPS * ref2["Om"].sum()
        assert abs(r["EcRPA"][m] - ref2["EcRPA"]) <= tol2, m
