"""The (T) operands at large v (k_triples_av has a workgroup per 4 x 4 block of virtuals and 8 of k: 17 million at
v = 1300, more than a launch along one axis takes).

24 of the virtuals carry integrals and amplitudes, spread over the whole range: the energy is that of the problem of these
24 alone, which the oracle gives.  Tolerance: split-BF16x3 3e-5, as for the other (T) tests."""
import numpy as np
import pytest

from helpers import random_amplitudes, random_df
from oracle import rccsd as R
from oracle import triples as TT

pytestmark = pytest.mark.gpu


def test_triples_v1300():
    import fermihip
    o, v, Q, m = 2, 1300, 6, 24
    print(f"triples o={o} v={v}", flush=True)
    eo, ev, Boo, Bov, Bvv = random_df(o, m, Q, 11)
    T1, T2 = random_amplitudes(o, m, 11)
    ref = TT.rccsdpt_ijk(T1, T2, R.build_moints(Boo, Bov, Bvv), eo, ev)
    at = np.concatenate([[0, 1, 7, 8, 31, 32], np.linspace(40, v - 12, m - 12).astype(int), np.arange(v - 6, v)])
    E = np.linspace(0.1, 3.0, v)
    E[at] = ev
    bov, bvv, t1, t2 = np.zeros((Q, o, v)), np.zeros((Q, v, v)), np.zeros((o, v)), np.zeros((o, o, v, v))
    bov[:, :, at] = Bov
    bvv[:, at[:, None], at[None]] = Bvv
    t1[:, at] = T1
    t2[:, :, at[:, None], at[None]] = T2
    c = fermihip.Context(0)
    c.set_df(eo, E, Boo, bov, bvv)
    e = c.triples(t1, t2, prec_mode=2)
    c.close()
    print(f"  rel {abs(e - ref) / abs(ref):.1e}", flush=True)
    assert abs(e - ref) < 3e-5 * abs(ref)
