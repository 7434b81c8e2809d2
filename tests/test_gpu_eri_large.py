"""Coulomb integrals of more pairs than one launch of k_eri takes (fh_integrals.hip, for_launches).

Tolerance: relative 1e-12, as for the other integral tests."""
import numpy as np
import pytest

from helpers import relerr
from oracle import integrals as I
from test_gpu_eri_classes import shell

pytestmark = pytest.mark.gpu


def test_more_workgroups_than_a_launch_takes():
    """(mu nu|P) of 2900 s functions and one fitting function: 4 206 450 pairs, a workgroup of 1024 threads each, where a
    launch takes 4 194 303.  Against the closed form, its normalisation from the oracle."""
    import fermihip
    from scipy.special import erf
    n, a, g = 2900, 0.8, 1.3
    print(f"eri {n} s functions", flush=True)
    xyz = np.random.default_rng(7).uniform(-3.0, 3.0, (n, 3))
    C = np.array([0.2, -0.1, 0.3])
    orb, aux = [shell(0, [a], [1.0], x) for x in xyz], [shell(0, [g], [1.0], C)]
    c = fermihip.Context(0)
    got = c.eri_2e3c(fermihip.Basis(orb), fermihip.Basis(aux))[:, :, 0]
    c.close()
    p = 2 * a
    d2 = ((xyz[:, None] - xyz[None]) ** 2).sum(2)
    T = p * g / (p + g) * (((xyz[:, None] + xyz[None]) / 2 - C) ** 2).sum(2)
    ref = np.exp(-a / 2 * d2) * np.sqrt(np.pi / T) / 2 * erf(np.sqrt(T))
    pick = [0, 1, 1450, n - 1]
    k = I.eri3c([orb[i] for i in pick], aux)[:, :, 0] / ref[np.ix_(pick, pick)]
    assert relerr(k, np.full((4, 4), k[0, 0])) < 1e-12
    assert relerr(got, k[0, 0] * ref) < 1e-12
