"""Calls that clear a device buffer have cleared it when they return: what the next call writes to it stays."""
import ctypes as C

import numpy as np
import pytest

import bayesrrcmd_amd as brr
from _data import make_bw_problem, make_problem

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


def test_num_record_of_the_next_sweep(gpu_lib):
    """brr_hip_record_num clears the record; the sweep right behind it fills it, also while the null stream is busy with
    another program part's work (here about 20 ms of fills)."""
    pr = make_problem(500, 200, seed=5, causal_frac=0.05)
    eps, sc = brr.bayesr_init(pr.y, 1, 2, 7)
    order = np.arange(pr.m, dtype=np.uint32)
    u, z = brr.marker_uz(3, 0, 0, pr.m)
    hip, other, size = C.CDLL("libamdhip64.so"), C.c_void_p(), 4 << 30
    got = []
    with brr.HipSweep(pr.n, pr.m, 2, 1, brr.LAYOUT_DENSE_2BIT) as h:
        h.upload_dense(pr.bed, pr.lut)
        h.set_model(np.array([0.001]))
        assert hip.hipMalloc(C.byref(other), C.c_size_t(size)) == 0
        for busy in (0, 20):
            h.set_state(eps, np.zeros(pr.m), np.zeros(pr.m, np.int32))
            h.set_scalars(sc["mu"], sc["sigmaE"], sc["epsilon_sum"], sc["sigmaG"], sc["pi"])
            for _ in range(busy):
                assert hip.hipMemsetAsync(other, 0, C.c_size_t(size), None) == 0
            h.record_num(True)
            h.sweep(order, u, z)
            got.append(h.get_num())
        assert hip.hipDeviceSynchronize() == 0 and hip.hipFree(other) == 0
    assert np.all(got[0] != 0) and np.array_equal(got[0], got[1])
