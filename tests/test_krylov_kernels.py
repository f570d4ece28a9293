"""GMRES over vector lengths at the edges of the solvers' chunks and basis sizes at
the edges of their vector groups: the residual of the solution, formed with the
step kernels and numpy, is the one the solver reports and stops at."""
import numpy as np
import pytest

from spectraldoublediffusiveconvection_amd import device as dev, newton

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# 3 N: 240 (one short chunk), 768 and 1024 + 8 (whole updates, one past a chunk),
# 3 * 1024 (whole chunks), 4416; restart: 1, 8, 9, 17 and 60 vectors
@pytest.mark.parametrize("K,Nr,restart", [(10, 9, 60), (32, 9, 8), (44, 9, 9), (128, 9, 17),
                                          (64, 24, 60), (10, 9, 1)])
def test_gmres_residual(K, Nr, restart):
    """The Arnoldi residual estimate holds to rounding: 1e-10 of the
    right-hand side (the estimate's own target is 1e-6)."""
    plan = dev.Plan.build(K, Nr, 0.35, 5e-3, 1.0, 1 / 15.0)
    k = newton.Krylov(plan, restart=restart)
    n = 3 * K * (Nr - 1)
    rng = np.random.default_rng(n + restart)
    X = torch.as_tensor(1e-3 * rng.standard_normal(n), device="cuda")
    b = torch.as_tensor(rng.standard_normal(n), device="cuda")
    x, info = k.gmres(X, b, 2700.0, 500.0, rtol=1e-6, max_restarts=2)
    Jx = plan.step_linearized(x[None], X[None], 2700.0, 500.0)[0] - x
    res = float(torch.linalg.norm(b - Jx)) / float(torch.linalg.norm(b))
    reported = info["residual"] / float(torch.linalg.norm(b))
    assert abs(res - reported) < 1e-10, (res, reported)
    assert res < 1.0 + 1e-9 and (not info["converged"] or res < 1.0001e-6)
    # and again: the same steps and bits
    again, info2 = k.gmres(X, b, 2700.0, 500.0, rtol=1e-6, max_restarts=2)
    assert torch.equal(again, x) and info2["iterations"] == info["iterations"]
    k.close()
    plan.close()
