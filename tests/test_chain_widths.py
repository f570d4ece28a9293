"""The launch shapes of the chains (Matrix_Operators.py:1033-1086, 1115-1194) give
the same bits: chain_segment N_fm/2, so that every plan here runs them."""
import numpy as np
import pytest

from oracle import sddc_oracle as O
from spectraldoublediffusiveconvection_amd import device as dev, operators as ops

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
PAR = dict(d=0.35, dt=5e-3, Pr=1.0, Tau=1 / 15.0)
WIDTHS = (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 16)


# 1, 2, 3 and 4 wavefronts of radial points; rows and radial points that fill their
# tiles (512, 33) and do not; 512/40 in the widths that its tuning entries use
@pytest.mark.parametrize("K,Nr,widths", [(64, 20, WIDTHS), (64, 33, WIDTHS), (64, 40, WIDTHS),
                                         (34, 65, WIDTHS), (512, 40, (1, 9, 16))])
def test_chain_widths_same_bits(K, Nr, widths):
    """Every launch shape of the chains: batches that fill no workgroup, some, and
    most of the last one step to the same bits, as does a graph of two parts, and
    instances of them to the oracle within 1e-12 (a back substitution 1e-14)."""
    op, nr = ops.build(K, Nr, **PAR), Nr - 1
    o = O.build_operators(K, Nr, PAR["d"], PAR["dt"], PAR["Pr"], PAR["Tau"])
    rng = np.random.default_rng(K + Nr)
    X = torch.as_tensor(1e-3 * rng.standard_normal((37, 3 * K * nr)), device="cuda")
    g = torch.as_tensor(rng.standard_normal((13, K * nr)), device="cuda")
    Ra = torch.linspace(2500.0, 9000.0, 37, dtype=torch.float64, device="cuda")
    first = None
    for w in widths:
        got = []
        for B in (1, 4, 5, 13, 37):
            p = dev.Plan(op, max_batch=B, tuning={"chain_segment": K // 2, "solve_instances": w})
            assert p.tuning()["chain_segment"] == K // 2
            got.append(p.step(X[:B], Ra[:B], 500.0, nsteps=2).cpu().numpy())
            if B == 13:
                got += [p.bsub(g, f).cpu().numpy() for f in range(3)]
            p.close()
        p = dev.Plan(op, max_batch=37, tuning={"chain_segment": K // 2, "solve_instances": w,
                                               "sub_batches": 2})
        x = X.clone()
        gr = p.graph(x, Ra, 500.0, nsteps=2)
        gr.launch()
        got.append(x.cpu().numpy())
        gr.close()
        p.close()
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[-1], got[-2]), w
        if first is None:
            first = got
        for a, b in zip(got, first):
            assert np.array_equal(a, b), w
    refs = [O.a4_bsub(g[12].cpu().numpy(), o.Linv_A4, o.D2_A4, o.IR4_A4, o.IR2_A4, K, nr,
                      PAR["Pr"] * PAR["dt"], False)]
    refs += [O.nab2_bsub(g[12].cpu().numpy(), L, K, nr, h, False)
             for L, h in ((o.Linv_T, PAR["dt"]), (o.Linv_S, PAR["Tau"] * PAR["dt"]))]
    for f, ref in zip(first[4:7], refs):
        assert np.linalg.norm(f[12] - ref) < 1e-14 * np.linalg.norm(ref)
    for b in (0, 36):
        ref = X[b].cpu().numpy()
        for _ in range(2):
            ref = O.step(ref, o, float(Ra[b]), 500.0)
        assert np.linalg.norm(first[-1][b] - ref) < 1e-12 * np.linalg.norm(ref), b
