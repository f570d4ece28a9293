"""The algorithmic bytes of the step's stages (profiling.stage_bytes), which the
bench line's bandwidths divide by."""
from types import SimpleNamespace

from spectraldoublediffusiveconvection_amd import profiling


def test_solve_counts_each_operator_block_once():
    """Right-hand sides in, states and suffix sums out, and one block inverse per
    mode and field: the chains stream no other blocks."""
    K, nr = 512, 39
    plan = SimpleNamespace(N_fm=K, nr=nr, precision_name="mixed")
    for B in (1, 64):
        arrays = (3 + 3 + 1) * B * K * nr
        assert profiling.stage_bytes(plan, B, 4) == 8 * (arrays + 3 * K * nr * nr)
