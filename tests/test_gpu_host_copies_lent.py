"""The pinned buffers of copies in chunks, lent by one context to another (IdlePool, fh_host.h): contexts in turn and in
threads of their own, sizes for which they are made, found at hand and not used; exact copies throughout."""
import threading

import pytest

from helpers import random_df

pytestmark = pytest.mark.gpu


def round_trips(o, v, seed, out):
    import fermihip
    try:
        eo, ev, Boo, Bov, Bvv = random_df(o, v, 4, seed)
        c = fermihip.Context(0)
        c.set_df(eo, ev, Boo, Bov, Bvv)
        for _ in range(3):
            T1, T2 = c.guess(0)
            e = c.energy()
            assert c.energy(T1, T2) == e
        c.close()
        out.append(e)
    except Exception as x:   # reported by the caller
        out.append(x)


def test_contexts_in_turn_and_in_threads():
    sizes = [(8, 100), (16, 127), (10, 90), (20, 110), (9, 85), (17, 122)]   # 4.9 to 36.9 MiB
    print("host copies lent", flush=True)
    alone = []
    for k, (o, v) in enumerate(sizes):
        round_trips(o, v, k, alone)
    together = [[] for _ in sizes]
    th = [threading.Thread(target=round_trips, args=(o, v, k, together[k])) for k, (o, v) in enumerate(sizes)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert [x[0] for x in together] == alone, (alone, together)
