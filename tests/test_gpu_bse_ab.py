"""GPU: the device-built BSE matrices and the two spins' side-by-side solves at the
smallest pair counts, around the 256-element blocks of the kernel and with frozen
orbitals, against the CPU restatement (oracle/gw_oracle.py rgw_phbse).

Tolerance: both sides solve Z = T^T (A + B) T with backward errors of a few nS eps |Z|
(nS <= 64, |Z| < 100, Om > 0.4): 10 nS eps |Z| / (2 Om) = 2e-11 in an energy; EcBSE sums
2 nS of them: 2e-9."""
import numpy as np
import pytest

from oracle import gw_oracle as go

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nO, nC, nR", [(2, 1, 0, 0), (17, 1, 0, 0), (18, 1, 0, 0), (7, 3, 1, 1), (9, 8, 0, 0),
                                           (16, 8, 0, 0)])
@pytest.mark.parametrize("tda", [False, True])
def test_bse_matrices_at_the_edges(n, nO, nC, nR, tda):
    from quack_amd import dfgen, gw
    print("bse", n, nO, nC, nR, tda, flush=True)
    e, B, _ = dfgen.synthetic_df(n, nO, 3 * n, seed=n + 100 * nO)
    B = np.asarray(B).reshape(3 * n, n, n)
    eri = np.einsum("Ppr,Pqs->pqrs", B, B)
    eGW = e + np.where(np.arange(n) < nO, -0.1, 0.1)
    Ec, OmS, OmT = go.rgw_phbse(eri, e, eGW, nO, eta=0.05, TDA=tda, nC=nC, nR=nR)
    assert OmT.min() > 0.4 and OmS.max() < 10
    r = gw.RGW_phBSE(eri, e, eGW, nO, eta=0.05, TDA=tda, nC=nC, nR=nR)
    assert np.abs(r["OmS"] - OmS).max() < 2e-11
    assert np.abs(r["OmT"] - OmT).max() < 2e-11
    assert np.abs(r["EcBSE"] - Ec).max() < 2e-9
