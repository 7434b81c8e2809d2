"""Paths that other tests compare with themselves, against independent ones: the reduced-precision (T) at the (H2O)10 shape
against the FP64 kernels and in other chunks, fh_mp2_energy_noalloc against the oracle.

Tolerances: split-BF16x3 3e-5 and FP32 1e-6 as for the other (T) tests; the same products in other chunks 1e-12 (their
FP64 partial sums add up in another order); DF-MP2 1e-12."""
import numpy as np
import pytest

from helpers import random_df
from oracle.rmp2 import rmp2_energy_df
from test_zz_no_alloc import DevBuf, _hip

pytestmark = pytest.mark.gpu


def test_triples_precisions_and_chunks_water10(monkeypatch):
    import fermihip
    from fermihip import synth
    print("(T) precisions and chunks water10 (40,190,840)", flush=True)
    eo, ev, Boo, Bov, Bvv, _, _ = synth.water_cluster_like(10, 0)
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    T1, T2 = c.guess()
    T1 = 0.01 * np.random.default_rng(5).standard_normal(T1.shape)
    e = [c.triples(T1, T2, prec_mode=p) for p in (0, 1, 2)]
    monkeypatch.setenv("FERMIHIP_TRIPLES_CHUNK_MB", "96")
    f = [c.triples(T1, T2, prec_mode=p) for p in (1, 2)]
    c.close()
    print(f"  fp32 {abs(e[1] / e[0] - 1):.1e} bf16x3 {abs(e[2] / e[0] - 1):.1e} chunks {abs(f[0] / e[1] - 1):.1e} "
          f"{abs(f[1] / e[2] - 1):.1e}", flush=True)
    assert abs(e[1] - e[0]) < 1e-6 * abs(e[0])
    assert abs(e[2] - e[0]) < 3e-5 * abs(e[0])
    assert abs(f[0] - e[1]) < 1e-12 * abs(e[1])
    assert abs(f[1] - e[2]) < 1e-12 * abs(e[2])


@pytest.mark.parametrize("o,v,Q", [(1, 1, 1), (5, 19, 84), (9, 17, 32), (53, 33, 17), (40, 190, 840)])
def test_noalloc_mp2_matches_oracle(o, v, Q):
    import fermihip
    print(f"noalloc DF-MP2 against the oracle o={o} v={v} Q={Q}", flush=True)
    hip = _hip()
    eo, ev, _, Bov, _ = random_df(o, v, Q, o + v + Q, 0.05)
    ref = rmp2_energy_df(Bov, eo, ev)
    c = fermihip.Context(0)
    bufs = [DevBuf(hip, x) for x in (eo, ev, Bov, [np.nan])]
    try:
        assert hip.hipDeviceSynchronize() == 0
        rc = c.L.fh_mp2_energy_noalloc(c.h, o, v, Q, *[b.p for b in bufs])
        assert rc == 0, c.L.fh_last_error().decode()
        assert abs(float(bufs[3].read()[0]) - ref) < 1e-12 * abs(ref)
    finally:
        for b in bufs:
            b.free()
        c.close()
