"""GPU: the full solve whose launch sequences are captured and replayed (qk_set_graphs), which
is the one for eigenvectors of a split-precision contraction: replay after replay equals
eager launches bit for bit.  Six solves with vectors alternate the handle's two matrix
buffers (one is the G0W0's), so either graph is replayed at least once after its capture,
with eager self-energy sweeps and a values-only solve in between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["mixed", "mixed2"])
def test_split_solves_replayed(systems, precision):
    from quack_amd import gw
    print("split-precision replay, H10", precision, flush=True)
    s = systems["H10"]
    rng = np.random.default_rng(13)
    es = [s["eHF"] + 1e-3 * rng.standard_normal(s["eHF"].size) for _ in range(5)]

    def run(graphs):
        gw.set_graphs(graphs)
        out = []
        with gw.GWEngine(s["nBas"], s["nOrb"], s["nO"]) as g:
            g.set_eri_ao(s["eri"], s["c"])
            g.set_precision(precision)
            g.set_eigensolver("sytrd")
            for k, ek in enumerate(es):
                g.screen(ek)
                out.append(g.sigma_at(ek, ek + 0.3, eta=0.05))
                if k == 2:
                    r = g.g0w0(s["eHF"])
                    out.append((r["eGW"], r["Om"]))
            assert g.eig_stats()["own_tridiagonal"] == 7
        return out

    try:
        eager = run(False)
        graph = run(True)
    finally:
        gw.set_graphs(False)
    for k, (a, b) in enumerate(zip(eager, graph)):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), k
