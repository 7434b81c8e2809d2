"""The Coulomb integral kernels (k_pair_e, k_eri) against the oracle where they can go wrong: every Hermite order of
bra and ket, contractions longer than a workgroup's wavefronts and than k_pair_e's 16 primitive pairs, more than 64
kets of one order, arguments of the Boys function around its table's points and beyond its end at 32.

Tolerance: relative 1e-12, as for the other integral tests."""
import numpy as np
import pytest

from helpers import relerr
from oracle import integrals as I

pytestmark = pytest.mark.gpu


def shell(l, exps, coefs, center):
    return {"l": l, "center": np.asarray(center, float), "exps": list(exps), "coefs": list(coefs)}


@pytest.mark.parametrize("spherical", [True, False])
def test_contracted_classes(spherical):
    import fermihip
    print(f"eri classes spherical={spherical}", flush=True)
    orb = [shell(0, [180.0, 31.0, 8.2, 2.4, 0.7, 0.25], [0.05, 0.2, 0.4, 0.4, 0.2, 0.1], (0, 0, 0)),
           shell(2, [1.7, 0.5], [0.6, 0.5], (0.3, -0.2, 0.4)), shell(1, [4.0, 1.1, 0.4], [0.2, 0.5, 0.4], (0, 1.1, -0.7)),
           shell(2, [1.2], [1.0], (0, 1.1, -0.7))]
    aux = [shell(l, [2.1 / (l + 1)], [1.0], (0.2, 0.5, 0.1 * l)) for l in (3, 2, 1, 0)] + \
          [shell(1, [3.0, 0.8], [0.3, 0.8], (0, 0, 9.0))]
    c = fermihip.Context(0)
    bs, ab = fermihip.Basis(orb, spherical), fermihip.Basis(aux, spherical)
    assert relerr(c.eri_2e3c(bs, ab), I.eri3c(orb, aux, spherical)) < 1e-12
    assert relerr(c.eri_2e2c(ab), I.eri2c(aux, spherical)) < 1e-12
    got = c.eri_2e4c(bs)
    assert relerr(got, I.eri4c(orb, spherical)) < 1e-12
    for p in ((1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1)):
        assert np.array_equal(got, got.transpose(p)) or relerr(got, got.transpose(p)) < 1e-14
    c.close()


def test_many_kets_and_boys_range():
    """70 s fitting functions a distance d apart, T = al d^2 from 0 over the table's half steps to far beyond 32."""
    import fermihip
    print("eri kets and Boys range", flush=True)
    orb = [shell(0, [1.0], [1.0], (0, 0, 0)), shell(1, [1.0], [1.0], (0, 0, 0)), shell(2, [1.0], [1.0], (0, 0, 0))]
    # pair exponent 2, fitting exponent 2: al = 1, T = d^2
    T = np.concatenate([np.arange(0, 40) / 16.0, 31.9375 + np.arange(-6, 10) / 32.0, np.geomspace(40.0, 900.0, 14)])
    aux = [shell(0, [2.0], [1.0], (0, 0, np.sqrt(t))) for t in T] + [shell(3, [2.0], [1.0], (0, np.sqrt(t), 0)) for t in (3.0, 32.0)]
    c = fermihip.Context(0)
    got = c.eri_2e3c(fermihip.Basis(orb), fermihip.Basis(aux))
    ref = I.eri3c(orb, aux)
    c.close()
    assert got.shape[2] == 70 + 14
    assert relerr(got, ref) < 1e-12
    # the s column alone, element by element
    assert np.abs(got[0, 0, :70] / ref[0, 0, :70] - 1).max() < 1e-12
