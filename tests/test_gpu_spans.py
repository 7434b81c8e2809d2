"""The times of fh_stats when a call has many more spans than wait to be read back (Spans, fh_host.h)."""
import pytest

from helpers import random_amplitudes, random_df

pytestmark = pytest.mark.gpu


def test_spans_of_many_chunks(monkeypatch):
    """(T) in chunks of 1 MiB: 2 of the 1520 triples each at v = 40, four spans a chunk. Each is counted once, and the
    spans inside one another add up to no more than the one around them."""
    import fermihip
    o, v = 20, 40
    print(f"spans o={o} v={v}", flush=True)
    eo, ev, Boo, Bov, Bvv = random_df(o, v, 12, 1)
    T1, T2 = random_amplitudes(o, v, 1)
    c = fermihip.Context(0)
    c.set_df(eo, ev, Boo, Bov, Bvv)
    e = c.triples(T1, T2)
    monkeypatch.setenv("FERMIHIP_TRIPLES_CHUNK_MB", "1")
    before = c.stats()["phases"]
    assert abs(c.triples(T1, T2) - e) < 1e-12 * abs(e)
    after = c.stats()["phases"]
    c.close()
    ms = {}
    for k in ("triples", "triples_gemm", "triples_w_first", "triples_w_slices", "triples_energy"):
        ms[k] = after[k]["ms"] - before[k]["ms"]
        assert after[k]["calls"] - before[k]["calls"] == (1 if k == "triples" else 760)
    print("  ms", {k: round(x, 2) for k, x in ms.items()}, flush=True)
    assert 0 < ms["triples_w_first"] + ms["triples_w_slices"] <= ms["triples_gemm"] * 1.001
    assert 0 < ms["triples_gemm"] + ms["triples_energy"] <= ms["triples"] * 1.001
