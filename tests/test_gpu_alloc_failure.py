"""A residual whose first call runs out of device memory while it makes its constants: the next call makes them, and is
held to the oracle at 1e-12 as in the other residual tests."""
import ctypes
import gc

import pytest

from helpers import random_amplitudes, random_df, relerr
from oracle import rccsd as R
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


def test_ladder_operand_after_a_failed_call():
    """o = 4, v = 120: with 950 MB free the ladder's operand (843 MB) is allocated and its workspace (207 MB) is not."""
    import fermihip
    o, v, Q, left = 4, 120, 8, 950 << 20
    print(f"allocation failure o={o} v={v}", flush=True)
    eo, ev, Boo, Bov, Bvv = random_df(o, v, Q, 2)
    T1, T2 = random_amplitudes(o, v, 2)
    n1, n2 = R.update_amp(T1, T2, R.build_moints(Boo, Bov, Bvv), eo, ev)
    hip = _hip()
    gc.collect()   # contexts of other tests
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    c.energy(T1, T2)   # the integral blocks
    ballast = []

    def take(n):
        p = ctypes.c_void_p()
        if hip.hipMalloc(ctypes.byref(p), n) != 0:
            hip.hipGetLastError()
            return None
        return p

    try:
        # all but 6 GB, then ever smaller pieces, each only where `left` is still to be had with it
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        ballast.append(take(a.value - (6 << 30)))
        n = 2 << 30
        while n >= 16 << 20:
            p = take(n + left)
            if p is None:
                n //= 2
                continue
            hip.hipFree(p)
            ballast.append(take(n))
        p = take(left)
        assert p is not None
        hip.hipFree(p)
        with pytest.raises(fermihip.FermiException, match="out of device memory"):
            c.update_amp(T1, T2)
    finally:
        for p in ballast:
            hip.hipFree(p)
    a1, a2 = c.update_amp(T1, T2)
    c.close()
    assert relerr(a1, n1) < 1e-12 and relerr(a2, n2) < 1e-12
