"""GPU: the AO to MO block of a batch, whose products run side by side in groups of
molecules, against the engine of one molecule: strides wider than the arrays, dropped
functions with frozen orbitals, and a batch of one full group and a remainder (N = 100:
eight molecules a group).

Tolerance: both sum every product in the same order; the energies differ by the rounding of
the batched eigensolve and sums, a few nS eps of terms below 10 Ha: 1e-11."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nmol, N, n, nO, nC, nR, pad", [(2, 5, 5, 1, 0, 0, 3), (3, 20, 17, 4, 1, 2, 0),
                                                         (9, 100, 100, 8, 0, 0, 0)])
def test_groups_match_one_molecule(nmol, N, n, nO, nC, nR, pad):
    import torch
    from quack_amd import gw
    print("batch aotomo", nmol, N, n, flush=True)
    g = torch.Generator("cuda").manual_seed(N)
    eri = torch.zeros(nmol, N ** 4 + pad, dtype=torch.float64, device="cuda")
    c = torch.zeros(nmol, N * n + pad, dtype=torch.float64, device="cuda")
    e = np.stack([np.concatenate([np.linspace(-1.5 - 0.01 * m, -0.5, nO), np.linspace(0.3, 4.0 + 0.1 * m, n - nO)])
                  for m in range(nmol)])
    for m in range(nmol):
        B = torch.randn(2 * N, N, N, generator=g, dtype=torch.float64, device="cuda") * (0.05 / N ** 0.5)
        B = (B + B.transpose(1, 2)).reshape(2 * N, N * N).contiguous()
        chem = (B.T.contiguous() @ B).reshape(N, N, N, N)  # (pr|qs) at [p, r, q, s]
        eri[m, :N ** 4] = chem.permute(3, 1, 2, 0).reshape(-1)  # p fastest, then q, r, s
        q, _ = torch.linalg.qr(torch.randn(N, n, generator=g, dtype=torch.float64, device="cuda"))
        c[m, :N * n] = q.T.reshape(-1)
        del B, chem
    torch.cuda.synchronize()
    with gw.GWBatch(nmol, N, n, nO, nC=nC, nR=nR) as b:
        b.set_eri_ao_device(eri.data_ptr(), N ** 4 + pad, c.data_ptr(), N * n + pad)
        r = b.g0w0(e, eta=0.1)
    with gw.GWEngine(N, n, nO, nC=nC, nR=nR) as h:
        for m in range(nmol):
            h.set_eri_ao_device(eri[m].data_ptr(), c[m].data_ptr())
            ref = h.g0w0(e[m], eta=0.1)
            assert np.abs(r["eGW"][m] - ref["eGW"]).max() < 1e-11, m
            assert abs(r["EcRPA"][m] - ref["EcRPA"]) < 1e-11, m
