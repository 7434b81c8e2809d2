"""The residual's kernels against the oracle at the edges of their tiles: o and v around the 32 x 32 blocks of
k_amp_forms / k_t2_numerator / k_vv_pairs, o > v, one of each, and packed ladders whose GEMM is cut along K (32 x 32
tiles at v = 40, 64 x 64 at v = 50).

Tolerance: as for the other residual tests, relative 1e-12."""
import pytest

from helpers import random_amplitudes, random_df, relerr
from oracle import rccsd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v", [(1, 1), (1, 34), (33, 3), (32, 5), (7, 32), (5, 33), (31, 2), (6, 40), (9, 50)])
def test_residual_tile_edges(o, v):
    import fermihip
    print(f"residual tiles o={o} v={v}", flush=True)
    eo, ev, Boo, Bov, Bvv = random_df(o, v, 12, o + 2 * v)
    m = R.build_moints(Boo, Bov, Bvv)
    T1, T2 = random_amplitudes(o, v, o + v)
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    g1, g2 = c.update_amp(T1, T2)
    r1, r2 = R.update_amp(T1, T2, m, eo, ev)
    c.close()
    assert relerr(g1, r1) < 1e-12
    assert relerr(g2, r2) < 1e-12
