"""The packing of cohorts into launches: the chain that takes longest comes first, by what a block and a beta change cost."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import test_gpu_cohorts as tc
from _data import make_problem

pytestmark = pytest.mark.gpu


def test_longest_chain_is_packed_first(gpu_lib):
    # two chains of 5 blocks whose every beta changes, and one of 94 blocks with few changes, which takes longer (an
    # iteration of about 230 us against 430); two of the three fit a launch
    ms, rare = [300, 300, 6000], [0.01, 0.01, 0.99]
    hs, orders = [], []
    for q, m in enumerate(ms):
        pr = make_problem(8000 + 16 * q, m, seed=800 + q, causal_frac=0.002)
        h = tc.build(pr, tc.orc.RAGGED, q, workgroups=100)
        sc = h.get_scalars()
        h.set_scalars(sc["mu"], sc["sigmaE"], sc["epsilon_sum"], np.array([1e-4]),
                      np.array([rare[q]] + [(1 - rare[q]) / 3] * 3))
        orders.append(tc.orders_for(m, q, 1))
        h.run_chain(tc.SEED, q, 0, orders[q])
        hs.append(h)
    rate = [h.stats()["changes"] / m for h, m in zip(hs, ms)]
    assert min(rate[:2]) > 0.9 and rate[2] < 0.03
    P = [h.stats()["workgroups"] for h in hs]
    assert sum(P) > 256 and sum(P[1:]) <= 256, P
    _, rep = brr.run_cohorts(hs, tc.SEED, 1, orders, chains=[0, 1, 2])
    assert rep["launches"] == 2 and rep["launch_of"][2] == 0, rep
    for h in hs:
        h.close()
