"""Large copies between the device and host memory (copy_staged: pinned chunks of 2 MiB, four threads) through entry
points that copy T2 both ways: just under its 4 MiB, just over, and many chunks with a ragged last one.

The copies are exact, so the energy of the amplitudes that came back equals that of those on the device; the guess itself
is held to the oracle at 1e-13, as in the other guess tests."""
import numpy as np
import pytest

from helpers import random_df, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v", [(8, 90), (8, 91), (13, 61), (16, 77)])
def test_t2_round_trip(o, v):
    import fermihip
    print(f"host copies o={o} v={v}: {8 * (o * v) ** 2} bytes", flush=True)
    eo, ev, Boo, Bov, Bvv = random_df(o, v, 9, o * v)
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    T1, T2 = c.guess(0)
    m = {"OVOV": np.einsum("Qia,Qjb->iajb", Bov, Bov, optimize=True)}
    D = eo[:, None, None, None] + eo[None, :, None, None] - ev[None, None, :, None] - ev[None, None, None, :]
    assert relerr(T2, m["OVOV"].transpose(0, 2, 1, 3) / D) < 1e-13
    e = c.energy()
    assert c.energy(T1, T2) == e
    assert c.energy(T1, np.ascontiguousarray(T2)) == e
    c.close()
