"""Gradients of the warm-start MLP at widths and batches off every tile: rows
padded to 8, transposes of ragged batches, products split over K and not, and
a smaller batch after a larger one (workspaces keep no stale padding)."""
import sys

import numpy as np
import pytest

from gpusim2grid_amd import _capi
from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,H,n_out,batches", [
    (3, 5, 2, (1, 9)),              # everything inside one tile's corner
    (236, 100, 236, (130, 33)),     # pads of 4
    (602, 256, 602, (300, 77)),     # pads of 6, 2 split input products
    (1993, 96, 131, (65,)),         # odd rows, a split of 7 over one tile
    (64, 512, 4097, (257, 511)),    # one column past the tiles of the output
])
def test_gradients_at_ragged_widths(n_in, H, n_out, batches):
    net = _capi.Mlp(n_in, H, n_out, seed=2)
    p0 = M.init_params(n_in, H, n_out, seed=2)
    rng = np.random.default_rng(n_in)
    for k in ("b1", "b2", "b3"):
        p0[k] = rng.normal(0, 0.1, p0[k].shape)
    net.set_params(p0)
    p = {k: np.asarray(v, np.float32).astype(np.float64) for k, v in p0.items()}
    for m in batches:
        print(f"mlp widths {n_in}-{H}-{n_out} m={m}", flush=True)
        sys.stdout.flush()
        X = rng.normal(size=(m, n_in)).astype(np.float32)
        T = rng.normal(size=(m, n_out)).astype(np.float32)
        L, g = net.loss_grad(X, T)
        Lref, gref = M.grad(p, X.astype(np.float64), T.astype(np.float64), bf16_ops=True)
        # the bounds of the other gradient tests: the same bf16 roundings, and
        # one-ulp flips of rounded hidden values
        assert abs(L - Lref) < 1e-3 * Lref
        for k in M.NAMES:
            err = np.linalg.norm(g[k] - gref[k]) / max(np.linalg.norm(gref[k]), 1e-30)
            assert err < 2e-2, (k, err)
        Y = net.forward(X)
        Yb, _ = M.forward(p, X.astype(np.float64), bf16_ops=True)
        assert np.abs(Y - Yb).max() < 5e-3 * np.abs(Yb).max()


def test_two_steps_equal_one_network_trained_alike():
    """Steps on device arrays equal steps on host arrays bit for bit (the targets
    are read in place, the copies refreshed by the step itself)."""
    import torch
    n_in, H, n_out, m = 602, 256, 602, 100
    rng = np.random.default_rng(8)
    X = rng.normal(size=(2, m, n_in)).astype(np.float32)
    T = rng.normal(size=(2, m, n_out)).astype(np.float32)
    a, b = (_capi.Mlp(n_in, H, n_out, seed=6) for _ in range(2))
    Xd, Td = torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda()
    torch.cuda.synchronize()
    for net in (a, b):
        net.set_grad_clip(0.3)
    for k in range(2):
        la = a.train_step(X[k], T[k], 1e-3)
        lb = b.train_step_device(Xd[k].data_ptr(), Td[k].data_ptr(), m, 1e-3)
        assert la == lb
    pa, pb = a.get_params(), b.get_params()
    for k in pa:
        np.testing.assert_array_equal(pa[k], pb[k])
    np.testing.assert_array_equal(a.forward(X[0]), b.forward(X[0]))
