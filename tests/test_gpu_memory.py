"""What a context holds on the device: the eigensolver's rocBLAS workspace is given back when an allocation would fail."""
import ctypes

import numpy as np
import pytest

from helpers import random_scf
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


def test_failed_allocation_gives_the_eigensolver_workspace_back():
    """(ij|kl) of 1000 occupied orbitals (8 TB) is refused (-4); what the device has free is then again what it had before
    the SCF, but for the small buffers of the two problems."""
    import fermihip
    hip = _hip()

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    o, v = 1000, 20
    print("memory of the eigensolver", flush=True)
    S, H, b = random_scf(200, 60, 1)
    opts = fermihip.ScfOptions(scf_max_iter=2)
    c = fermihip.Context(0)
    c.rhf(S, H, b, 20, options=opts)   # loads the library's kernels, which stay
    c.close()
    c = fermihip.Context(0)
    f0 = free()
    r0 = c.rhf(S, H, b, 20, options=opts)[0]
    f1 = free()
    c.set_df(np.linspace(-2.0, -1.0, o), np.linspace(1.0, 2.0, v), *[np.full((1, p, q), 1e-3) for p, q in ((o, o), (o, v), (v, v))])
    with pytest.raises(fermihip.FermiException, match="out of device memory"):
        c.prepare()
    f2 = free()
    print(f"  free before, with, after: {f0 >> 20}, {f1 >> 20}, {f2 >> 20} MiB", flush=True)
    assert f0 - f2 <= 16 << 20
    r1 = c.rhf(S, H, b, 20, options=opts)[0]
    c.close()
    assert r1["energy"] == r0["energy"]
