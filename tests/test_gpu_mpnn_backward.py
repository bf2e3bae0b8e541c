"""The network's backward kernels at the edges of their tiles (32 cells a wave on the way back, 16 a
wave and 256 blocks in the weight gradients) and for each width of the neighbour lists."""
import numpy as np
import pytest

import oracle.mpnn as om
from dopamine_amd.mpnn import LearnedPreconditioner
from test_gpu_mpnn import channel_poisson, random_params

pytestmark = pytest.mark.gpu


def widened(nbr, coef, w):
    """The same rows in w slots (the last ones empty)."""
    more = w - nbr.shape[0]
    return np.vstack([nbr, np.full((more, nbr.shape[1]), -1, nbr.dtype)]), np.vstack([coef, np.zeros((more, nbr.shape[1]))])


def chain_poisson(n):
    nbr = -np.ones((2, n), dtype=np.int32)
    nbr[0, 1:], nbr[1, :-1] = np.arange(n - 1), np.arange(1, n)
    coef = np.where(nbr >= 0, 1.0 + 0.1 * np.arange(n) % 7, 0.0)
    coef[0, 1:] = coef[1, :-1]
    return nbr, coef, coef.sum(axis=0) + 0.05


@pytest.mark.parametrize("shape,w", [((2, 1, 1), 4), ((33, 1, 1), 4), ((127, 1, 1), 4), ((5, 4, 3), 6), ((7, 5, 3), 8),
                                     ((9, 8, 7), 10), ((32, 16, 2), 6), ((41, 23, 19), 6)])
def test_weight_gradients_at_tile_edges(shape, w):
    nx, ny, nz = shape
    nbr, coef, diag = chain_poisson(nx) if ny * nz == 1 else channel_poisson(nx, ny, nz)
    nbr, coef = widened(np.asarray(nbr), np.asarray(coef), w)
    net, g = LearnedPreconditioner(nbr, coef, diag, capacity=1, seed=2), om.Graph(nbr, coef, diag)
    flat = random_params(21)
    net.params = flat
    wts = om.unflatten(flat.astype(np.float64))
    r = np.random.default_rng(8).standard_normal(g.diag.size)
    print(f"[gpu] mpnn backward {shape} w {w}", flush=True)
    loss, grad, hs = net.loss_grad(r, activations=True)
    L, grads = om.backward_from(wts, g, r, hs)
    assert abs(loss - L) <= 1e-5 * L
    gd = om.unflatten(grad)
    for k in om.PARAM_ORDER:  # FP32 rounding of the chain back, averaged over the cells
        assert np.linalg.norm(gd[k] - grads[k]) <= 2e-6 * np.linalg.norm(grads[k]), k
