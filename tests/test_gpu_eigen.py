"""The SCF's small eigensolver (fh_eigen.hip) through fh_rhf: sizes on both sides of its register tiles (32 .. 160) and of
its range (3 .. 160), against the oracle's SCF as in test_gpu_rhf (one iteration), and the overlap's inverse root on a
matrix that is tridiagonal or diagonal already (reflectors that are 1).

Tolerances: as test_gpu_rhf; orthonormality n 2^-52 times a factor of 100."""
import numpy as np
import pytest

from helpers import random_scf
from oracle import rhf as RH

pytestmark = pytest.mark.gpu


def run(S, H, b, nd):
    import fermihip
    n = S.shape[0]
    ref = RH.rhf(S, H, b, nd, 0.5, RH.Options(scf_max_iter=1))
    r = fermihip.RHF(S, H, b, nd, 0.5, options=fermihip.ScfOptions(scf_max_iter=1))
    print(f"eigen n={n}: dE {abs(r.energy - ref['energy']):.1e}", flush=True)
    assert abs(r.energy - ref["energy"]) < 1e-10 * abs(ref["energy"])
    assert np.max(np.abs(r.eps - ref["eps"])) < 1e-8
    assert np.max(np.abs(r.C @ np.diag(r.eps) @ r.C.T - ref["C"] @ np.diag(ref["eps"]) @ ref["C"].T)) < 1e-8
    assert np.max(np.abs(r.C.T @ S @ r.C - np.eye(n))) < 100 * n * 2.0**-52 * np.linalg.cond(S)


@pytest.mark.parametrize("n", [3, 4, 17, 31, 32, 33, 64, 65, 96, 97, 128, 129, 159, 160, 161])
def test_sizes(n):
    run(*random_scf(n, max(6, n // 2), n), max(1, n // 5))


@pytest.mark.parametrize("n", [5, 40])
def test_reflectors_that_are_one(n):
    _, H, b = random_scf(n, 8, n)
    run(np.eye(n), np.diag(np.linspace(-3.0, 2.0, n)) + 0.1 * (np.eye(n, k=1) + np.eye(n, k=-1)), 1e-3 * b, max(1, n // 5))
