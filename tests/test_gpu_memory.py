"""What a context holds on the device: the (T) without the constants of the CCSD residual, and the eigensolver's rocBLAS
workspace given back when an allocation would fail."""
import ctypes

import numpy as np
import pytest

from helpers import random_amplitudes, random_df, random_scf
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


def test_triples_holds_no_residual_constants(monkeypatch):
    """The peak of a (T) on new integrals, in doubles: B, the five blocks, T1 and T2, AV and Bcat twice each, (ia|jb) of
    which a second copy is made by blocks, a chunk of W of 1 MiB, tables under 2 MiB; no other o^2 v^2 tensor."""
    import fermihip
    o, v, Q = 40, 24, 30
    print(f"memory triples o={o} v={v}", flush=True)
    monkeypatch.setenv("FERMIHIP_TRIPLES_CHUNK_MB", "1")
    eo, ev, Boo, Bov, Bvv = random_df(o, v, Q, 3)
    T1, T2 = random_amplitudes(o, v, 3)
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    c.triples(T1, T2)
    n2, nd = (o * v) ** 2, (o + v + 7) // 8 * 8
    need = Q * (o + v) ** 2 + o**4 + o**3 * v + 2 * n2 + o * v**3 + n2 + 2 * v * v * o * nd + 2 * nd * v * o * o + 2 * n2
    peak = c.stats()["pool_peak_bytes"]
    c.close()
    print(f"  peak {peak / 8 / n2:.2f} o^2 v^2, needed {need / n2:.2f}", flush=True)
    assert peak < 8 * need + (3 << 20) + 0.3 * 8 * n2


def test_prepare_leaves_no_constants_to_the_first_residual():
    """fh_prepare makes what the residual keeps. At o = v the tensors are o^4: five blocks, the ladder's two operands (one
    (1 + 1/v)^2 / 2), the residual's six others and B, 3 x 30 o^2; tables and rounding under a tenth."""
    import fermihip
    o = v = 24
    print(f"memory prepare o={o} v={v}", flush=True)
    c = fermihip.Context(0)
    c.set_df(*random_df(o, v, 30, 4))
    c.prepare()
    peak = c.stats()["pool_peak_bytes"] / (8 * o**4)
    c.close()
    print(f"  peak {peak:.1f} o^4", flush=True)
    assert 0 <= peak - (12 + (1 + 1 / v) ** 2 / 2 + 90 / v**2) < 0.1


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
