"""Cohort calls whose Gram rows take several steps: the same chains, bit for bit, as one iteration per call, with all
counters, through the graph and launched directly. (Three cohorts of about 20,000 markers: 8 iterations fill a step's
524,288 rows.)"""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import test_gpu_cohorts as tc
from _data import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [True, False], ids=["graph", "direct"])
@pytest.mark.parametrize("precision", [brr.PRECISION_FP64, brr.PRECISION_FP32_REFRESH], ids=["fp64", "fp32"])
def test_several_steps_equal_single_iterations(gpu_lib, precision, graph):
    iters = 10                       # two steps of 5
    sizes = [(400, 20_000, tc.orc.DENSE, 0.0), (700, 21_003, tc.orc.RAGGED, 0.01), (300, 20_500, tc.orc.DENSE, 0.01)]
    probs = [make_problem(n, m, seed=700 + q, causal_frac=0.001, maf=(0.05, 0.5), miss=miss)
             for q, (n, m, _, miss) in enumerate(sizes)]
    orders = [tc.orders_for(pr.m, q, iters) for q, pr in enumerate(probs)]
    runs = []
    for step in (iters, 1):
        hs = [tc.build(pr, lay, q, precision) for q, (pr, (_, _, lay, _)) in enumerate(zip(probs, sizes))]
        hist, rounds, changes = [[] for _ in hs], np.zeros(len(hs), int), np.zeros(len(hs), int)
        for it in range(0, iters, step):
            out, rep = brr.run_cohorts(hs, tc.SEED, it, [o[it:it + step] for o in orders], chains=[0, 1, 2], graph=graph)
            assert rep["launches"] == 1
            for q, h in enumerate(hs):
                hist[q].append(out[q])
                rounds[q] += h.stats()["rounds"]
                changes[q] += h.stats()["changes"]
        runs.append(([np.concatenate(x) for x in hist], rounds, changes, [h.get_state() for h in hs],
                     [h.get_scalars() for h in hs]))
        for h in hs:
            h.close()
    (ha, ra, ca, sa, xa), (hb, rb, cb, sb, xb) = runs
    assert np.array_equal(ra, rb) and np.array_equal(ca, cb) and np.all(ca > 0)
    for q in range(len(probs)):
        assert np.array_equal(ha[q], hb[q]), q
        for k in sa[q]:
            assert np.array_equal(sa[q][k], sb[q][k]), (q, k)
        for k in ("mu", "sigmaE", "epsilon_sum", "v", "betasqn", "pi", "sigmaG"):
            assert np.array_equal(xa[q][k], xb[q][k]), (q, k)
        # and the chain that the context runs alone
        alone = tc.build(probs[q], sizes[q][2], q, precision)
        assert np.array_equal(alone.run_chain(tc.SEED, q, 0, orders[q]), ha[q]), q
        assert np.array_equal(alone.get_state()["eps"], sa[q]["eps"]), q
        alone.close()


def test_iteration_in_parts(gpu_lib):
    """More markers in all than a step may hold (8,388,608): each iteration in two parts of every cohort's blocks. One of
    the cohorts has a single block and so markers in one part only."""
    n, m, copies, iters = 64, 262_144 + 65, 32, 2
    pr = make_problem(n, m, seed=7, causal_frac=0.0001, maf=(0.3, 0.5))
    small = make_problem(200, 40, seed=8, causal_frac=0.1)
    rng = np.random.default_rng(4)
    probs = [pr] * copies + [small]
    ys = [rng.permutation(pr.y) for _ in range(copies)] + [small.y]

    images = [brr.bed_file_image(p.bed) for p in (pr, small)]

    def make(q):
        p = probs[q]
        h = brr.HipSweep(p.n, p.m, 4, 1, brr.LAYOUT_DENSE_2BIT)
        h.load_bed(images[q == copies], brr.LAYOUT_DENSE_2BIT)
        h.set_model(tc.S)
        eps, sc = brr.bayesr_init(ys[q], 1, 4, tc.SEED, chain=q)
        h.set_state(eps, np.zeros(p.m), np.zeros(p.m, np.int32))
        h.set_scalars(sc["mu"], sc["sigmaE"], sc["epsilon_sum"], sc["sigmaG"], sc["pi"])
        return h

    hs = [make(q) for q in range(len(probs))]
    big, few = tc.orders_for(m, 0, iters), tc.orders_for(small.m, 1, iters)
    orders = [big] * copies + [few]
    hists, rep = brr.run_cohorts(hs, tc.SEED, 0, orders, chains=list(range(len(hs))))
    assert rep["launches"] == 1
    for q in (0, copies - 1, copies):
        alone = make(q)
        assert np.array_equal(alone.run_chain(tc.SEED, q, 0, orders[q]), hists[q]), q
        sa, sb = alone.get_state(), hs[q].get_state()
        for k in sa:
            assert np.array_equal(sa[k], sb[k]), (q, k)
        xa, xb = alone.get_scalars(), hs[q].get_scalars()
        assert np.array_equal(xa["v"], xb["v"]) and np.array_equal(xa["betasqn"], xb["betasqn"])
        assert alone.stats()["rounds"] == hs[q].stats()["rounds"] and alone.stats()["changes"] == hs[q].stats()["changes"]
        alone.close()
    for h in hs:
        h.close()
