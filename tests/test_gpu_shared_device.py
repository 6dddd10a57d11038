"""GPU: the full solve where a launch whose workgroups wait for each other counts as given up
(a host-side switch: the launch itself ends normally), where such launches are switched off,
and as it is, against LAPACK (numpy) on the same matrix: strip back-transformation, GEMM
back-transformation (orders above 2048) and a matrix whose last columns alone fit the
registers (above 3072), with vectors checked through the self-energy.

The launch-per-column form rounds otherwise than the registers, which tells which one ran.
Tolerances: those of test_gpu_eigh.py."""
import numpy as np
import pytest

from test_gpu_eigh import om_tolerance, reference, system

pytestmark = pytest.mark.gpu


def check(r, ref, B, e, nO):
    assert (np.abs(r["Om"] - ref["Om"]) <= om_tolerance(ref)).all()
    assert np.abs(r["SigC"] - ref["SigC"]).max() <= 1e-10 * np.abs(ref["SigC"]).max()
    # the values-only solve at the quasiparticle energies
    ref2 = reference(r["eGW"], B, nO, False)
    tol2 = 0.5 * om_tolerance(ref2).sum() + len(ref2["Om"]) * np.finfo(float).eps * ref2["Om"].sum()
    assert abs(r["EcRPA"] - ref2["EcRPA"]) <= tol2


@pytest.mark.parametrize("nO,nV", [(7, 23), (12, 32), (26, 50), (41, 50), (56, 56)])
def test_engine(nO, nV):
    from quack_amd import gw
    n = nO + nV
    print("shared device", nO, nV, flush=True)
    e, B = system(nO, nV, nO * nV)
    ref = reference(e, B, nO, True)
    Om = {}
    with gw.GWEngine(n, n, nO) as g:
        g.set_eri_df(B)
        for mode in (0, 1, 2):
            g.set_shared_device(mode)
            r = g.g0w0(e, eta=0.1, linearize=True)
            check(r, ref, B, e, nO)
            Om[mode] = r["Om"]
        again = g.g0w0(e, eta=0.1, linearize=True)["Om"]  # what was given up is remembered
        g.set_shared_device(0)
        back = g.g0w0(e, eta=0.1, linearize=True)["Om"]
    assert not np.array_equal(Om[0], Om[1])
    assert np.array_equal(Om[1], Om[2]) and np.array_equal(Om[1], again) and np.array_equal(Om[0], back)


def test_batch():
    from quack_amd import gw
    print("shared device, batch", flush=True)
    nO, nV, nmol = 9, 19, 3
    n = nO + nV
    sys_ = [system(nO, nV, 50 + m) for m in range(nmol)]
    es = np.stack([e for e, _ in sys_])
    Om = {}
    with gw.GWBatch(nmol, n, n, nO) as b:
        for m, (_, B) in enumerate(sys_):
            chem = np.einsum("Ppq,Prs->pqrs", B, B, optimize=True)
            b.set_eri_mo(m, np.asfortranarray(chem.transpose(0, 2, 1, 3)))
        for mode in (0, 1, 2):
            b.set_shared_device(mode)
            r = b.g0w0(es, eta=0.1, linearize=True)
            for m, (e, B) in enumerate(sys_):
                check({k: r[k][m] for k in ("Om", "SigC", "eGW", "EcRPA")}, reference(e, B, nO, True), B, e, nO)
            Om[mode] = r["Om"]
    assert not np.array_equal(Om[0], Om[1]) and np.array_equal(Om[1], Om[2])


def test_refused_modes():
    from quack_amd import gw
    with gw.GWEngine(3, 3, 1) as g:
        for mode in (-1, 3):
            with pytest.raises(gw.QKError) as ex:
                g.set_shared_device(mode)
            assert ex.value.code == gw.QK_E_ARG
