"""Network kernels at cell counts below one row tile, off the tile's and the
padding's multiples, and above one tile per block of the backward grid
(40,320 cells: 630 tiles of 64 rows over 512 blocks): forward, loss and
every gradient against the oracle (test_gpu_gnn.py trains).

Tolerances as in test_gpu_gnn.py: BF16 rounding of GEMM inputs that differ in
the last FP32 bit, 1e-3 (forward, loss) and 2e-3 (gradients) in norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, dtype=np.float64) - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("core,ring,nslab", [(1, 1, 1), (2, 1, 3), (3, 1, 5), (8, 5, 30)])
def test_forward_and_gradient(tmp_path, core, ring, nslab):
    from nodals_amd import meshgen
    from nodals_amd._lib import Gnn, H8
    from oracle import gnn_oracle as G

    d = str(meshgen.write_pipe_case(tmp_path / "pipe", core=core, ring=ring, nslab=nslab))
    print(f"\n[gpu] GNN core={core} ring={ring} nslab={nslab}", flush=True)
    h = H8(["--mesh", d, "--max-outer", "10", "--verbose", "0"])
    g = Gnn(h, seed=3)
    graph = G.Graph(*h.gnn_graph()[:2])
    rng = np.random.default_rng(nslab)
    for rep in range(2):  # the second pass reuses the staged rows
        x = (rng.standard_normal((g.n, G.IN)) * 0.7).astype(np.float32)
        t = (rng.standard_normal(g.n) - 1.0).astype(np.float32)
        p = (g.params().astype(np.float64) + rng.standard_normal(g.params().size) * 0.05).astype(np.float32)
        g.set_params(p)
        yo, _ = G.forward(p.astype(np.float64), graph, x.astype(np.float64))
        assert rel(g.forward(x), yo) < 1e-3
        grad, loss = g.gradient(x, t)
        lo, go, _ = G.loss_and_grad(p.astype(np.float64), graph, x.astype(np.float64), t.astype(np.float64))
        assert abs(loss - lo) <= 1e-3 * lo
        for k, (o, s) in G.layout().items():
            if k != "_size":
                sl = slice(o, o + int(np.prod(s)))
                assert rel(grad[sl], go[sl]) < 2e-3, k
        assert np.array_equal(grad, g.gradient(x, t)[0])  # fixed order of every sum
    g.close()
    h.close()
