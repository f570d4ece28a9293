"""The nonlinear products over grid lengths on both sides of every column count
of the in-place kernels, and lengths that only the general ones take, against the
oracle (Matrix_Operators.py:743-898)."""
import numpy as np
import pytest

from oracle import sddc_oracle as O
from spectraldoublediffusiveconvection_amd import device as dev

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
PAR = (0.35, 5e-3, 1.0, 1 / 15.0)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# L = 3 N_fm / 2: 6, 60 | 72, 120 | 135 | 225, 243 | 300, 375 | 450, 486 | 540, 600 |
# 750, 810; 21 and 462 have factors above 5
@pytest.mark.parametrize("K", [4, 40, 48, 80, 90, 150, 162, 200, 250, 300, 324, 360, 400, 500, 540,
                               14, 308])
def test_products_at_length(K):
    """Tolerances of the parity tests: 1e-12 in float64, 2e-5 in mixed precision."""
    Nr, B = 9, 3
    n = 3 * K * (Nr - 1)
    rng = np.random.default_rng(K)
    decay = np.exp(-6.0 * np.arange(K) / K).repeat(Nr - 1)
    X, v = (rng.standard_normal((B, n)) * np.tile(decay, 3) for _ in range(2))
    o = O.build_operators(K, Nr, *PAR)
    tx, tv = (torch.as_tensor(a, device="cuda") for a in (X, v))
    for precision, tol in (("fp64", 1e-12), ("mixed", 2e-5)):
        p = dev.Plan.build(K, Nr, *PAR, precision=precision, max_batch=B)
        F = p.nlin_fx(tx).cpu().numpy()
        D = p.nlin_dfx(tv, tx).cpu().numpy()
        for b in (0, B - 1):
            assert rel(F[b], O.nlin_fx(X[b], o)) < tol, (precision, b)
            assert rel(D[b], O.nlin_dfx(v[b], X[b], o)) < tol, (precision, b)
        p.close()
