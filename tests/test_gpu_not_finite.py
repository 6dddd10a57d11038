"""GPU: matrices that are not finite (a NaN integral, orbital levels that cross, one bad
molecule of a batch) end in QK_E_EIG, and the next call on the same handle is right.
Orders: one Jacobi leaf without merges, one workgroup, several workgroups.

The divide and conquer used to run on such a matrix with merge positions that nobody had
written.  Tolerances of the good calls: those of test_gpu_eigh.py."""
import numpy as np
import pytest

from test_gpu_eigh import om_tolerance, reference, system

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3), (3, 43), (5, 41), (12, 32)]


def check_good(r, ref):
    assert (np.abs(r["Om"] - ref["Om"]) <= om_tolerance(ref)).all()
    assert np.abs(r["SigC"] - ref["SigC"]).max() <= 1e-10 * np.abs(ref["SigC"]).max()


def refused(gw, call):
    with pytest.raises(gw.QKError) as ex:
        call()
    assert ex.value.code == gw.QK_E_EIG


@pytest.mark.parametrize("nO,nV", SHAPES)
@pytest.mark.parametrize("mode", ["syevd", "sytrd"])
def test_engine(nO, nV, mode):
    from quack_amd import gw
    print("not finite, engine", nO, nV, mode, flush=True)
    e, B = system(nO, nV, nO * nV)
    ref = reference(e, B, nO, True)
    bad = B.copy()
    bad[0, 0, nO] = bad[0, nO, 0] = np.nan
    crossed = e.copy()
    crossed[[nO - 1, nO]] = crossed[[nO, nO - 1]]
    with gw.GWEngine(nO + nV, nO + nV, nO) as g:
        g.set_eigensolver(mode)
        for _ in range(2):
            g.set_eri_df(bad)
            refused(gw, lambda: g.g0w0(e, eta=0.1, linearize=True))
            refused(gw, lambda: g.evgw(e, eta=0.1, linearize=True))
            g.set_eri_df(B)
            refused(gw, lambda: g.g0w0(crossed, eta=0.1, linearize=True))
            check_good(g.g0w0(e, eta=0.1, linearize=True), ref)


@pytest.mark.parametrize("nO,nV", SHAPES)
def test_one_molecule_of_a_batch(nO, nV):
    from quack_amd import gw
    print("not finite, batch", nO, nV, flush=True)
    n, nmol = nO + nV, 3
    sys_ = [system(nO, nV, 7 + m) for m in range(nmol)]
    eris = [np.asfortranarray(np.einsum("Ppq,Prs->pqrs", B, B, optimize=True).transpose(0, 2, 1, 3)) for _, B in sys_]
    es = np.stack([e for e, _ in sys_])
    bad = eris[1].copy(order="F")
    bad[0, 0, nO, nO] = np.nan  # (pr|qs) at [p, q, r, s]: (0 nO|0 nO)
    crossed = es.copy()
    crossed[1, [nO - 1, nO]] = crossed[1, [nO, nO - 1]]
    with gw.GWBatch(nmol, n, n, nO) as b:
        for m in range(nmol):
            b.set_eri_mo(m, bad if m == 1 else eris[m])
        refused(gw, lambda: b.g0w0(es, eta=0.1, linearize=True))
        refused(gw, lambda: b.evgw(es, eta=0.1, linearize=True))
        b.set_eri_mo(1, eris[1])
        refused(gw, lambda: b.g0w0(crossed, eta=0.1, linearize=True))
        r = b.g0w0(es, eta=0.1, linearize=True)
    for m, (e, B) in enumerate(sys_):
        check_good({"Om": r["Om"][m], "SigC": r["SigC"][m]}, reference(e, B, nO, True))


@pytest.mark.parametrize("n", [5, 40, 170])
@pytest.mark.parametrize("tda", [False, True])
def test_phrlr(n, tda):
    """Good call: Om within n eps |Z| / Om of LAPACK's, |Z| < 40 and Om > 1: 1e-11."""
    from quack_amd import gw
    print("not finite, phRLR", n, tda, flush=True)
    rng = np.random.default_rng(n)
    A = 0.02 * rng.standard_normal((n, n))
    A = A + A.T + np.diag(np.linspace(2.0, 4.0, n))
    B = 0.005 * rng.standard_normal((n, n))
    B = B + B.T
    bad = A.copy()
    bad[n // 2, n // 2] = np.nan
    refused(gw, lambda: gw.phRLR(tda, bad, B))
    Om = gw.phRLR(tda, A, B)[1]
    if tda:
        want = np.linalg.eigvalsh(A)
    else:
        w, U = np.linalg.eigh(A - B)
        assert w[0] > 0.5
        T = U * np.sqrt(w)
        want = np.sqrt(np.linalg.eigvalsh(T.T @ (A + B) @ T))
    assert want[0] > 1.0 and want[-1] < 6.0
    assert np.abs(Om - want).max() < 1e-11
