"""Loss gradient of the T2-guess network against the oracle at the edges of its passes over the samples: one sample, one
workgroup's 16 columns and around, more than 16 x 1024 samples (longer column runs), the widest network, and sample
counts on both sides of the weight gradients' cut along K.

Tolerance per parameter block: 1e-4 of its largest element (FP32 sums), as for the other gradient test."""
import numpy as np
import pytest

from oracle import mlp as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,n", [(128, 1), (32, 15), (64, 16), (128, 17), (1, 40), (256, 200), (64, 383), (64, 384), (128, 16385),
                                 (32, 20001)])
def test_gradient_edges(h, n):
    import fermihip
    print(f"mlp gradient edges h={h} n={n}", flush=True)
    rng = np.random.default_rng(h + n)
    p = (0.3 * rng.standard_normal(M.nparams(h))).astype(np.float32)
    X = rng.standard_normal((n, 6)).astype(np.float32)
    T = (1.0 + rng.standard_normal(n)).astype(np.float32)
    net = fermihip.Mlp(hidden=h)
    net.set_params(p)
    L, g = net.loss_grad(X, T)
    Lr, gr = M.loss_grad(p.astype(np.float64), h, X.astype(np.float64), T.astype(np.float64))
    assert abs(L - Lr) < 1e-5 * abs(Lr)
    o = M.offsets(h)
    sizes = {"W1": 6 * h, "W2": h * h, "W3": h * h, "b4": 1}
    for k in ("W1", "b1", "W2", "b2", "W3", "b3", "w4", "b4"):
        blk = slice(o[k], o[k] + sizes.get(k, h))
        assert np.max(np.abs(g[blk] - gr[blk])) < 1e-4 * np.max(np.abs(gr[blk])) + 1e-9, k
