"""The solve form of a sweep's classes: on both sides of each line of the rule,
and against the oracle's steps."""
import numpy as np
import pytest

from oracle import sddc_oracle as O
from spectraldoublediffusiveconvection_amd import batching

torch = pytest.importorskip("torch")
EIGEN = {"chain_segment": 8, "solve_instances": 1, "sub_batches": 1}


def test_form_of_a_class():
    def form(N_fm, tuning):
        return batching.Sweep._fewer_launches((N_fm, 20), tuning)["chain_segment"]
    assert form(64, EIGEN) == 32 and form(256, EIGEN) == 128 and form(258, EIGEN) == 8
    chains = dict(EIGEN, chain_segment=64, solve_instances=9)
    assert batching.Sweep._fewer_launches((128, 20), chains) is chains


@pytest.mark.gpu
@pytest.mark.parametrize("classes,each,precision,chains", [(6, 2, "mixed", True), (5, 1, "mixed", False),
                                                           (6, 11, "mixed", False),
                                                           (6, 1, "fp64", False)])
def test_sweep_of_many_small_classes(classes, each, precision, chains):
    """Tolerances: those of the sweep's test (mixed 2e-5, float64 1e-12)."""
    class Table:
        def lookup(self, key, B, precision):
            return dict(EIGEN)
    sizes = [(258 if i == 0 else 98 + 12 * i, 12 + i) for i in range(classes)]
    rng = np.random.default_rng(classes + each)
    insts = []
    for K, Nr in sizes * each:
        x = rng.standard_normal(3 * K * (Nr - 1))
        insts.append(dict(N_fm=K, N_r=Nr, d=0.35, dt=5e-3, Pr=1.0, Tau=1 / 15.0,
                          Ra=float(rng.uniform(2500, 3000)), Ra_s=500.0,
                          X0=1e-3 * x / np.linalg.norm(x)))
    sw = batching.Sweep(insts, precision=precision, tuning_table=Table())
    for (K, *_), c in sw.classes.items():
        assert (c.plan.tuning()["chain_segment"] == K // 2) == (chains and K <= 256), K
    g = sw.graph(nsteps=3)
    g.launch()
    got = sw.states()
    g.close()
    for i in range(classes):
        inst = insts[i]
        o = O.build_operators(*batching.class_key(inst))
        x = inst["X0"]
        for _ in range(3):
            x = O.step(x, o, inst["Ra"], inst["Ra_s"])
        e = np.linalg.norm(got[i] - x) / np.linalg.norm(x)
        assert e < (2e-5 if precision == "mixed" else 1e-12), (i, e)


@pytest.mark.gpu
@pytest.mark.parametrize("classes,each,precision,chains", [(6, 1, "fp64", True), (5, 1, "fp64", False),
                                                           (6, 11, "fp64", False),
                                                           (6, 1, "mixed", True)])
def test_sweep_without_table_entries(classes, each, precision, chains):
    """The same lines for classes that the table has no entry for: a float64 sweep
    of many small classes waits for its launches as a mixed one does."""
    sizes = [(258 if i == 0 else 98 + 12 * i, 12 + i) for i in range(classes)]
    rng = np.random.default_rng(classes + each)
    insts = []
    for K, Nr in sizes * each:
        x = rng.standard_normal(3 * K * (Nr - 1))
        insts.append(dict(N_fm=K, N_r=Nr, d=0.35, dt=5e-3, Pr=1.0, Tau=1 / 15.0,
                          Ra=float(rng.uniform(2500, 3000)), Ra_s=500.0,
                          X0=1e-3 * x / np.linalg.norm(x)))

    class Table:
        def lookup(self, key, B, precision):
            return None
    for table in (None, Table()):
        sw = batching.Sweep(insts, precision=precision, tuning_table=table)
        for (K, *_), c in sw.classes.items():
            assert (c.plan.tuning()["chain_segment"] == K // 2) == (chains and K <= 256), K
        g = sw.graph(nsteps=2)
        g.launch()
        got = sw.states()
        g.close()
        for i in range(classes):
            o = O.build_operators(*batching.class_key(insts[i]))
            x = insts[i]["X0"]
            for _ in range(2):
                x = O.step(x, o, insts[i]["Ra"], insts[i]["Ra_s"])
            e = np.linalg.norm(got[i] - x) / np.linalg.norm(x)
            assert e < (2e-5 if precision == "mixed" else 1e-12), (i, e)
