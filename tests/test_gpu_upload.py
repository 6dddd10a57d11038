"""GPU: the (pq|jb) block gathered from a host array through the pinned ring arrives bit
for bit: with X + Y the unit matrix, the excitation densities are the block itself (the
products are x * 1 and x * 0).  One pair, a block below one slot, one of several turns of
the ring with a remainder, and frozen orbitals at both ends."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nO, nC, nR", [(2, 1, 0, 0), (9, 4, 1, 2), (17, 16, 0, 0), (41, 7, 1, 3), (41, 7, 0, 0)])
def test_block_of_the_active_pairs(n, nO, nC, nR):
    from quack_amd import gw
    print("block", n, nO, nC, nR, flush=True)
    eri = np.random.default_rng(n + nC).standard_normal((n, n, n, n))
    o, v = nO - nC, n - nR - nO
    rho = gw.RGW_excitation_density(eri.ravel(order="F"), np.eye(o * v), n, nO, nC=nC, nR=nR)
    blk = eri[:, nC:nO, :, nO:n - nR].transpose(0, 2, 1, 3).reshape(n, n, o * v)  # [p, q, b + v j]
    assert np.array_equal(rho, blk)
