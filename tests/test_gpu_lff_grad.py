"""Training gradient at the edges of its chunks (64 samples) and its grid (256
workgroups), against FP64 reverse mode; rows kept between calls of other sizes."""
import numpy as np
import pytest

import blitzar_amd as B
from oracle import mlp

pytestmark = pytest.mark.gpu


def test_gradient_at_chunk_and_grid_edges():
    rng = np.random.default_rng(1)
    p = (0.3 * rng.standard_normal(mlp.NP)).astype(np.float32)
    with B.OctreeHip(64) as s:
        for n in (16385, 63, 64, 65, 1, 16384, 33000):
            X = rng.normal(size=(n, mlp.NF)).astype(np.float32)  # the pad inputs too
            Y = rng.normal(size=(n, mlp.NO)).astype(np.float32)
            g, L = s.lff_gradient(X, Y, p)
            Lr, gr = mlp.loss_grad(p.astype(np.float64), X.astype(np.float64),
                                   Y.astype(np.float64))
            # FP32 sums: the tolerances of the one-chunk gradient test
            assert L == pytest.approx(Lr, rel=1e-5)
            assert np.linalg.norm(g - gr) <= 1e-5 * np.linalg.norm(gr), n
            assert np.abs(g - gr).max() <= 1e-4 * np.abs(gr).max(), n
            # each block of parameters on its own (a wrong bias hides in the whole)
            for a, b in zip(np.split(g, np.cumsum([2048, 64, 4096, 64, 192])),
                            np.split(gr, np.cumsum([2048, 64, 4096, 64, 192]))):
                assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b), n
            y = s.lff_forward(X[:5])
            assert y.shape == (min(n, 5), 3) and np.isfinite(y).all()


def test_forward_on_rows_kept_from_a_gradient():
    """The forward pass reads its own rows and writes behind them, whatever an
    earlier call of another size left in the row buffer."""
    rng = np.random.default_rng(2)
    p = (0.3 * rng.standard_normal(mlp.NP)).astype(np.float32)
    X = rng.normal(size=(20001, mlp.NF)).astype(np.float32)
    y64 = mlp.forward(p.astype(np.float64), X.astype(np.float64))
    scale = np.sqrt(np.mean(y64 * y64))
    with B.OctreeHip(64) as s:
        s.lff_set_params(p)
        for n, m in ((333, 5), (64, 20001), (20001, 1), (70, 333), (20001, 20001)):
            G = rng.normal(size=(n, mlp.NF)).astype(np.float32)
            s.lff_gradient(G, np.zeros((n, mlp.NO), np.float32), -p)
            y = s.lff_forward(X[:m])
            # BF16 inference: the tolerance of the forward pass on fresh rows
            assert y.shape == (m, 3) and np.abs(y - y64[:m]).max() <= 5e-2 * scale, (n, m)
