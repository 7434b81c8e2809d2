"""The fused guess inference beyond 2^31 amplitudes (a workgroup per 128 of them: more than a launch along one axis takes).

A network whose output is its last bias adds c = y_scale b4 to every amplitude; with one vector B_ia for the integrals the
energy is then the MP2 guess's plus c (sum B)^2. Tolerance: the network's output is FP32, c (sum B)^2 2^-23, and the energies'
rounding 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_guess_beyond_2_31_amplitudes():
    import fermihip
    o, v = 128, 364
    assert (o * v) ** 2 > 2**31
    print(f"learned guess o={o} v={v}", flush=True)
    rng = np.random.default_rng(3)
    B = rng.uniform(0.0, 0.01, (1, o, v))
    c = fermihip.Context(0)
    c.set_df(np.linspace(-2.0, -1.0, o), np.linspace(0.5, 3.0, v), np.zeros((1, o, o)), B, np.zeros((1, v, v)))
    c.guess(0, copy_out=False)
    e0 = c.energy()
    net = fermihip.Mlp(128)
    p = np.zeros(net.num_params, np.float32)
    p[-1] = 0.75
    net.set_params(p)
    net.x_mean, net.x_scale, net.y_scale = np.zeros(6, np.float32), np.ones(6, np.float32), 0.5
    c.set_t2_model(net, np.zeros((o, o)))
    c.guess(1, copy_out=False)
    e1 = c.energy()
    c.close()
    net.close()
    add = 0.375 * B.sum() ** 2
    print(f"  MP2 {e0:.6f} learned {e1:.6f} expected {e0 + add:.6f}", flush=True)
    assert abs(e1 - e0 - add) < 2.0**-23 * add + 1e-12 * (abs(e0) + add)
