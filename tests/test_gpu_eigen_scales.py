"""The SCF's small eigensolver on two blocks whose coupling is far below the others' scale (two molecules far apart):
the squares of a coupling column are then denormal or zero.  As in test_gpu_eigen, against the oracle's SCF of one
iteration, with its tolerances; the coupling itself is far below them."""
import numpy as np
import pytest

from helpers import random_scf
from test_gpu_eigen import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 24, 70])
@pytest.mark.parametrize("coupling", [1e-140, 1e-158, 1e-161, 2e-162, 1e-170, 1e-306, 1e-315])
def test_weakly_coupled_blocks(n, coupling):
    print(f"eigen blocks n={n} coupling {coupling:.0e}", flush=True)
    S, H, b = random_scf(n, max(6, n // 2), n)
    k = n // 2
    far = np.ones((n, n))
    far[:k, k:] = far[k:, :k] = coupling
    S, H, b = S * far, H * far, b * far
    run(S, H, b, max(1, n // 5))
