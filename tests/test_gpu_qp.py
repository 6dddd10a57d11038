"""GPU: the graphical QP solve on both sides of the size where it runs in one
launch (an orbital's excitation densities up to 4 MB), at sizes that leave
waves, lanes and rows of that launch without work.

The Newton iteration stops at |w - eHF - Sigma(w)| <= 1e-6 and steps once more,
so the residual at its result, with Sigma from the chunked sweep
(qk_gw_sigma_at), is below 1e-6 for every orbital that stopped.
"""
import numpy as np
import pytest

from test_gpu_eigh import system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nO,nV", [(1, 1), (1, 3), (1, 64), (5, 13), (8, 32), (9, 36), (20, 110), (32, 115)])
def test_newton_residual(nO, nV):
    from quack_amd import gw
    print("newton residual", nO, nV, flush=True)
    e, B = system(nO, nV, nO * nV)
    with gw.GWEngine(nO + nV, nO + nV, nO) as g:
        g.set_eri_df(B)
        r = g.g0w0(e, eta=0.1)
        it = g.qp_iters()
        g.screen(e)
        s, ds = g.sigma_at(e, r["eGW"], eta=0.1)
    ok = it < 64
    assert ok.all() and (it >= 1).all()
    assert np.abs(r["eGW"] - e - s).max() <= 1e-6
    # Z is the last step's 1 / (1 - dSigma), at a point within 2e-6 of the result
    assert np.abs(r["Z"] - 1.0 / (1.0 - ds)).max() <= 1e-4
