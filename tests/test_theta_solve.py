"""The solves in the eigenbasis of the theta operator, at the sizes where their
tiles, pairs and mode groups end, against the oracle's back substitutions
(Matrix_Operators.py:1033-1086, 1115-1194)."""
import numpy as np
import pytest

from oracle import sddc_oracle as O
from spectraldoublediffusiveconvection_amd import device as dev, operators as ops

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
PAR = dict(d=0.35, dt=5e-3, Pr=1.0, Tau=1 / 15.0)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# n = N_fm/2 rows per parity: one pair of tiles (24, 32), a row past it (33), a
# partial mode group (50, 75), several pairs (150, 256, 300); radial sizes of one
# to four column groups, odd and even; batches around the groups of 4 and 8
# instances and on both sides of the lone-tile rule.
@pytest.mark.parametrize("K,Nr,B", [(48, 9, 1), (64, 17, 3), (66, 20, 9), (100, 34, 4), (150, 65, 5),
                                    (300, 49, 8), (512, 40, 13), (528, 25, 2)])
@pytest.mark.parametrize("sym", [False, True])
def test_theta_solve(K, Nr, B, sym):
    """Tolerances: those of the chains' tests (1e-14 for a back substitution,
    to whose bound the plan holds the eigenbasis; 1e-12 for a step)."""
    o = O.build_operators(K, Nr, PAR["d"], PAR["dt"], PAR["Pr"], PAR["Tau"])
    p = dev.Plan(ops.build(K, Nr, **PAR), symmetric=sym, max_batch=B,
                 tuning={"chain_segment": 8})
    nr = Nr - 1
    rng = np.random.default_rng(K + Nr + B)
    g = rng.standard_normal((B, K * nr)) * np.logspace(0, -3, K).repeat(nr)[None, :]
    h = (PAR["Pr"] * PAR["dt"], PAR["dt"], PAR["Tau"] * PAR["dt"])
    for field in range(3):
        f = p.bsub(torch.as_tensor(g, device="cuda"), field).cpu().numpy()
        for b in range(B):
            if field == 0:
                ref = O.a4_bsub(g[b], o.Linv_A4, o.D2_A4, o.IR4_A4, o.IR2_A4, K, nr, h[0], sym)
            else:
                Linv = o.Linv_T if field == 1 else o.Linv_S
                ref = O.nab2_bsub(g[b], Linv, K, nr, h[field], sym)
            assert rel(f[b], ref) < 1e-14, (field, b)
    X = 1e-3 * rng.standard_normal((B, 3 * K * nr))
    Y = p.step(torch.as_tensor(X, device="cuda"), 2700.0, 500.0, nsteps=2).cpu().numpy()
    for b in sorted({0, B // 2, B - 1}):
        ref = X[b]
        for _ in range(2):
            ref = O.step(ref, o, 2700.0, 500.0, symmetric=sym)
        assert rel(Y[b], ref) < 1e-12, b
    p.close()


def test_other_operators_keep_the_chains():
    """Blocks that are no polynomials in the theta operator: the plan solves
    with the chains, which take any block inverses."""
    K, Nr, B = 128, 20, 3
    o = O.build_operators(K, Nr, PAR["d"], PAR["dt"], PAR["Pr"], PAR["Tau"])
    op = ops.build(K, Nr, **PAR)
    scale = 1.0 + 0.1 * np.arange(K)[:, None, None]
    op.Linv_T = np.ascontiguousarray(op.Linv_T * scale)
    p = dev.Plan(op, max_batch=B, tuning={"chain_segment": 8})
    nr = Nr - 1
    g = np.random.default_rng(0).standard_normal((B, K * nr))
    f = p.bsub(torch.as_tensor(g, device="cuda"), 1).cpu().numpy()
    for b in range(B):
        assert rel(f[b], O.nab2_bsub(g[b], o.Linv_T * scale, K, nr, PAR["dt"])) < 1e-14, b
    p.close()
