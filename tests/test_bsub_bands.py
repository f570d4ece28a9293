"""The psi, T and S back substitutions of right-hand sides confined to single rows
and bands of rows, at the default form of the plan's solves, against the oracle's
recurrences (Matrix_Operators.py:1033-1086, 1115-1194)."""
import numpy as np
import pytest

from oracle import sddc_oracle as O
from spectraldoublediffusiveconvection_amd import device as dev, operators as ops

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
PAR = dict(d=0.35, dt=5e-3, Pr=1.0, Tau=1 / 15.0)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def bands(K):
    """(first, past the last) rows of one parity."""
    n = K // 2
    rows = [(r, r + 1) for r in (0, 2, 12, 16, 24, 32, 48, n - 1)]
    return rows + [(b, e) for b, e in ((8, 12), (16, 24), (22, 30), (32, n))]


@pytest.mark.parametrize("K,Nr", [(128, 30), (300, 48), (512, 40)])
@pytest.mark.parametrize("parity", [0, 1])
def test_band_limited_back_substitution(K, Nr, parity):
    """1e-14: the bound of every back substitution test.  The values above the
    band are zero, exactly."""
    nr, cuts = Nr - 1, bands(K)
    B = len(cuts)
    o = O.build_operators(K, Nr, PAR["d"], PAR["dt"], PAR["Pr"], PAR["Tau"])
    p = dev.Plan(ops.build(K, Nr, **PAR), max_batch=B)
    rng = np.random.default_rng(K + parity)
    g = np.zeros((B, K, nr))
    for b, (lo, hi) in enumerate(cuts):
        g[b, parity + 2 * lo:parity + 2 * hi:2] = rng.standard_normal((hi - lo, nr))
    g = g.reshape(B, -1)
    h = (PAR["Pr"] * PAR["dt"], PAR["dt"], PAR["Tau"] * PAR["dt"])
    for field in range(3):
        f = p.bsub(torch.as_tensor(g, device="cuda"), field).cpu().numpy()
        for b, (lo, hi) in enumerate(cuts):
            if field == 0:
                ref = O.a4_bsub(g[b], o.Linv_A4, o.D2_A4, o.IR4_A4, o.IR2_A4, K, nr, h[0], False)
            else:
                ref = O.nab2_bsub(g[b], o.Linv_T if field == 1 else o.Linv_S, K, nr, h[field],
                                  False)
            assert rel(f[b], ref) < 1e-14, (field, lo, hi)
            assert not f[b].reshape(K, nr)[parity + 2 * hi:].any(), (field, lo, hi)
    p.close()
