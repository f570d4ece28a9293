"""The form of the solves that a plan reports is the one it runs."""
import numpy as np
import pytest

from spectraldoublediffusiveconvection_amd import device as dev, operators as ops

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
PAR = dict(d=0.35, dt=5e-3, Pr=1.0, Tau=1 / 15.0)


# the sizes of tests/test_theta_solve.py
@pytest.mark.parametrize("K,Nr", [(48, 9), (64, 17), (66, 20), (100, 34), (150, 65), (300, 49),
                                  (512, 40), (528, 25)])
def test_eigenbasis_is_reported(K, Nr):
    p = dev.Plan(ops.build(K, Nr, **PAR), tuning={"chain_segment": 8})
    assert p.tuning()["chain_segment"] == 8
    p.close()


@pytest.mark.parametrize("field", ["Linv_A4", "Linv_T", "Linv_S"])
@pytest.mark.parametrize("segment", [0, 8])
def test_fallback_is_reported(field, segment):
    """Blocks that are no polynomials in the theta operator: the chains."""
    K, Nr = 128, 20
    op = ops.build(K, Nr, **PAR)
    scale = 1.0 + 0.1 * np.arange(K)[:, None, None]
    setattr(op, field, np.ascontiguousarray(getattr(op, field) * scale))
    p = dev.Plan(op, tuning={"chain_segment": segment})
    assert p.tuning()["chain_segment"] == K // 2
    p.close()


def test_few_radial_points_report_the_chains():
    p = dev.Plan(ops.build(128, 8, **PAR), tuning={"chain_segment": 8})   # 7 interior points
    assert p.tuning()["chain_segment"] == 64
    p.close()
