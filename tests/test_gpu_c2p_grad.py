"""The loss gradient of the learned guess on the GPU (k_mlp_batch,
k_mlp_sum) at the row counts where its tiling can go wrong: one row, the
edges of a 32-row tile, one tile per workgroup (4096) and more tiles than
workgroups, against the float64 oracle."""
import numpy as np
import pytest

from disco_amd import c2p_model
from oracle import c2pnet

pytestmark = pytest.mark.gpu

# A gradient entry is a float32 sum over n rows of products of float32
# activations, each a sum of up to 64 products: relative to the sum of the
# terms' magnitudes its error is below (64 + 64 + 40) eps from the three
# layers and the tile, workgroup and block sums (at most 32 + 8 + 128 terms
# each), eps = 2^-24: 336 eps = 2e-5; cancellation between terms is bounded
# by comparing with the gradient's 2-norm.
TOL = 2e-5


@pytest.mark.parametrize("n", [1, 31, 32, 33, 1000, 4096, 4097, 20000])
def test_gradient_matches_float64(n):
    from test_c2p_train import _problem
    print(f"case dh_c2p_grad n={n}", flush=True)
    # normalised over at least 8 rows: one row has no spread
    p, X, Y = _problem(n=max(n, 8), seed=n)
    X, Y = X[:n], Y[:n]
    g, loss = c2p_model.grad(p, X, Y)
    g64, l64 = c2pnet.grad(p, X, Y)
    err = np.linalg.norm(g - g64) / np.linalg.norm(g64)
    print(f"  rel {err:.2e}, loss {abs(loss - l64) / l64:.2e}", flush=True)
    assert err < TOL
    assert abs(loss - l64) < TOL * l64
