"""GPU: products of a few tiles (the 32 x 32 matrix-core tile), through the excitation
densities rho(pq, m) = sum_jb (pq|jb) (X + Y)(m, jb): sizes below, at and just past a
multiple of the tile and of its 16-deep slabs.  Tolerance: K + 2 roundings of the terms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# nS = nO nV: 1, 8, 16, 20, 31, 32, 33, 48, 65
@pytest.mark.parametrize("n, nO", [(2, 1), (6, 2), (8, 4), (9, 4), (32, 1), (12, 4), (14, 3), (16, 4), (18, 13)])
def test_product_of_few_tiles(n, nO):
    from quack_amd import gw
    print("product", n, nO, flush=True)
    rng = np.random.default_rng(n)
    eri = rng.standard_normal((n, n, n, n))
    S = nO * (n - nO)
    x = rng.standard_normal((S, S))
    rho = gw.RGW_excitation_density(eri.ravel(order="F"), np.asfortranarray(x), n, nO)
    blk = eri[:, :nO, :, nO:].transpose(0, 2, 1, 3).reshape(n, n, S)
    ref = blk @ x.T
    bound = 2 * (S + 2) * np.finfo(float).eps * (np.abs(blk) @ np.abs(x).T)
    assert np.all(np.abs(rho - ref) <= bound)
