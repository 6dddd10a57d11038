"""GPU: phRLR of A and B that are not symmetric, which QuAcK's routine takes as they come (its
eigensolves read the upper triangles of A - B and of Z in the pairs' own basis),
against the CPU restatement, on either side of the eigensolver's leaf and
one-workgroup orders.

Tolerances: backward errors of a few n eps |Z| on either side, n <= 161, |Z| < 30, Om > 1,
2e-11 of an energy at most (the asymmetry moves them by more than 1e-4 from order 16 on); X +- Y are
checked mode by mode through gaps of more than 2e-3 in Z: 161 eps 30 / 2e-3 of a vector, 1e-9."""
import numpy as np
import pytest

from oracle import gw_oracle as go

pytestmark = pytest.mark.gpu


def matrices(n):
    rng = np.random.default_rng(n)
    A = 0.02 * rng.standard_normal((n, n)) + np.diag(np.linspace(2.0, 4.0, n))
    B = 0.02 * rng.standard_normal((n, n))
    return np.asfortranarray(A), np.asfortranarray(B)


@pytest.mark.parametrize("n", [1, 2, 16, 17, 50, 161])
@pytest.mark.parametrize("tda", [False, True])
def test_asymmetric(n, tda):
    from quack_amd import gw
    print("phRLR asymmetric", n, tda, flush=True)
    A, B = matrices(n)
    Ec0, Om0, XpY0, XmY0 = go.phRLR(tda, A, B)
    assert Om0[0] > 1.0 and Om0[-1] < 5.4
    if n > 2:
        sym = go.phRLR(tda, 0.5 * (A + A.T), 0.5 * (B + B.T))[1]
        assert np.abs(sym - Om0).max() > 1e-4
    Ec, Om, XpY, XmY = gw.phRLR(tda, A, B)
    assert np.abs(Om - Om0).max() < 2e-11
    assert abs(Ec - Ec0) < 2e-11 * n
    lam = Om0 if tda else Om0 ** 2
    gap = np.full(n, np.inf)
    if n > 1:
        d = np.diff(lam)
        gap = np.minimum(np.r_[np.inf, d], np.r_[d, np.inf])
    k = np.argmax(np.abs(XpY0), axis=1)
    sgn = np.sign(XpY[np.arange(n), k] * XpY0[np.arange(n), k])[:, None]
    on = gap > 2e-3
    assert on.sum() >= 0.8 * n
    assert np.abs(sgn * XpY - XpY0)[on].max() < 1e-9
    assert np.abs(sgn * XmY - XmY0)[on].max() < 1e-9
