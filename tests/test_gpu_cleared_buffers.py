"""Calls that clear a device buffer have cleared it when they return: what the next call writes to it stays."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
from _data import make_bw_problem

pytestmark = pytest.mark.gpu


def test_covariates_of_a_survival_model(gpu_lib):
    """X' failure of the covariates, formed by brr_hip_bw_set_fixed behind its clearing, decides their draws: the same
    draws in every context."""
    pr = make_bw_problem(2225, 10, seed=3)
    X = np.random.default_rng(4).normal(size=(pr.n, 2)).astype(np.float32)
    eps, sc = brr.bayesw_init(pr.y, pr.fail, pr.m, 3)
    draws = []
    for _ in range(60):
        with brr.HipBayesW(pr.n, pr.m, 3) as h:
            h.upload_ragged(pr.ragged)
            h.set_model(np.array([0.001, 0.01]), pr.fail)
            h.set_fixed(X)
            h.set_state(eps, np.zeros(pr.m), np.zeros(pr.m, np.int32))
            h.set_scalars(sc["mu"], sc["alpha"], sc["sigma_b"], sc["d"], sc["pi"])
            h.fixed_effects(5, 0)
            draws.append(h.get_theta())
    assert np.all(draws[0] != 0) and np.array_equal(draws, [draws[0]] * len(draws))
