"""The (T) W build's tiles and chunks (fh_triples.hip) against the oracle, through the C ABI: v around the tile and
block edges of the split-BF16x3 kernel (32-blocks, 64 MB tiles), of the FP64 / FP32 kernels (16-blocks, 32 .. 96
wide tiles) and of the padded k groups of 8, and chunk lengths that cut a run of k.

Tolerances (relative, as for the other (T) tests): FP64 1e-12; FP32 1e-6 (2^-23 per product); split-BF16x3 3e-5
(2^-16 per product)."""
import pytest

from helpers import random_amplitudes, random_df
from oracle import rccsd as R
from oracle import triples as TT

pytestmark = pytest.mark.gpu

BOUND = {0: 1e-12, 1: 1e-6, 2: 3e-5}


def run(o, v, seed, precs=(0, 1, 2)):
    import fermihip
    print(f"triples tiles o={o} v={v}", flush=True)
    eo, ev, Boo, Bov, Bvv = random_df(o, v, 12, seed)
    m = R.build_moints(Boo, Bov, Bvv)
    T1, T2 = random_amplitudes(o, v, seed)
    ref = TT.rccsdpt_ijk(T1, T2, m, eo, ev)
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    for prec in precs:
        e = c.triples(T1, T2, prec_mode=prec)
        if v == 1:  # a = b = c only: V cancels term by term (4 + 2 - 6), in the oracle up to its rounding
            assert e == 0.0 and abs(ref) < 1e-15
            continue
        print(f"  prec {prec}: rel {abs(e - ref) / abs(ref):.1e}", flush=True)
        assert abs(e - ref) < BOUND[prec] * abs(ref)
    c.close()


@pytest.mark.parametrize("o,v", [(2, 1), (3, 2), (2, 6), (4, 16), (3, 17), (5, 31), (3, 32), (4, 33), (3, 47), (2, 65), (3, 80),
                                 (2, 97), (3, 128), (2, 129), (2, 160), (2, 161), (2, 193), (9, 3)])
def test_triples_tile_edges(o, v):
    run(o, v, 3 * o + v)


@pytest.mark.parametrize("mb", ["1", "3"])
def test_triples_chunks(mb, monkeypatch):
    """Chunks of 1 or 3 MiB of W: at v = 30 4 and 14 slots (FP64), 9 and 29 (FP32), cutting the runs of k (up to 8)."""
    monkeypatch.setenv("FERMIHIP_TRIPLES_CHUNK_MB", mb)
    run(8, 30, 5)


@pytest.mark.parametrize("o,v", [(3, 4), (2, 5), (3, 20), (3, 29), (2, 46), (3, 78), (2, 100), (2, 196), (2, 203)])
def test_triples_last_panel(o, v):
    """W's planes lie in panels of 8 a: every v % 8, with the last panel alone, in a tile of its own and behind others."""
    run(o, v, 5 * o + v)
