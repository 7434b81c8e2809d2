"""The DF-MP2 pair kernel (fh_mp2.hip) against the oracle at the edges of its tiles (v around 32 and 64, blocks of 16), of
its pairs and of its K steps (naux around 16 and 32, odd).

Tolerance: relative 1e-12, as for the other DF-MP2 tests."""
import pytest

from helpers import random_df
from oracle.rmp2 import rmp2_energy_df

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,Q", [(1, 1, 1), (8, 16, 31), (9, 17, 32), (2, 31, 33), (7, 32, 64), (3, 33, 15), (17, 48, 16), (2, 63, 17),
                                   (9, 64, 5), (4, 65, 47), (8, 80, 48), (3, 97, 40), (2, 130, 21), (40, 3, 9), (53, 33, 17), (53, 64, 33), (31, 65, 15),
                                   (31, 97, 16), (31, 130, 31)])
def test_mp2_tile_edges(o, v, Q):
    import fermihip
    print(f"mp2 tiles o={o} v={v} Q={Q}", flush=True)
    eo, ev, _, Bov, _ = random_df(o, v, Q, o + v + Q)
    c = fermihip.Context(0)
    c.set_df(eo, ev, None, Bov, None)
    e, ref = c.mp2_energy(), rmp2_energy_df(Bov, eo, ev)
    c.close()
    assert abs(e - ref) < 1e-12 * abs(ref)
