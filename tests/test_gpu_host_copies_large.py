"""Copies to the device in chunks (copy_chunked): T2 of just under and just over 32 MiB, and with a ragged last chunk.

The copies are exact, so the energy of amplitudes that went to the host and back equals that of those on the device."""
import pytest

from helpers import random_df

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v", [(16, 127), (16, 129), (23, 101)])
def test_t2_to_the_device(o, v):
    import fermihip
    print(f"host copies o={o} v={v}: {8 * (o * v) ** 2} bytes", flush=True)
    eo, ev, Boo, Bov, Bvv = random_df(o, v, 5, o * v)
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    T1, T2 = c.guess(0)
    e = c.energy()
    assert c.energy(T1, T2) == e
    assert c.energy(T1, T2.copy(order="F")) == e
    c.close()
