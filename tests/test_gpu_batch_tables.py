"""Batched dense sweeps whose tables hold no number where no call points: a workgroup's residual tiles past its slice
look up no code of their own."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
import test_gpu_batch as tb
from _data import make_problem

pytestmark = pytest.mark.gpu


# slices of 1, 3 and 9 tiles of 16 individuals in kernels built for 4, 4 and 13 tiles (FP64) and 8, 8 and 16 (FP32)
@pytest.mark.parametrize("n,workgroups", [(500, 0), (500, 11), (1150, 8)])
@pytest.mark.parametrize("precision", [brr.PRECISION_FP64, brr.PRECISION_FP32], ids=["fp64", "fp32"])
def test_values_of_codes_that_do_not_occur(gpu_lib, n, workgroups, precision):
    pr = make_problem(n, 70, seed=n + workgroups, h2=0.5, causal_frac=0.1)
    T = 20
    os_ = tb.oracle_traits(pr, orc.DENSE, tb.phenotypes(pr, T, seed=3), 41)
    # a sweep over columns whose calls are nearly all missing first: it leaves its codes in local memory
    full = make_problem(4096, 70, seed=9, miss=0.9)
    before = tb.device_traits(full, orc.DENSE, tb.oracle_traits(full, orc.DENSE, tb.phenotypes(full, T, seed=3), 41),
                              workgroups=16)
    order = brr.shuffle(41, 0, 0, np.arange(pr.m, dtype=np.uint32))
    uz = [brr.marker_uz(41, 0, t, pr.m) for t in range(T)]
    u, z = np.stack([a for a, _ in uz], axis=1), np.stack([b for _, b in uz], axis=1)
    out = []
    for last in (0.0, np.nan, np.inf):
        before.sweep(order, u, z)
        lut = pr.lut.copy()
        lut[:, 3] = last
        h = tb.device_traits(pr, orc.DENSE, os_, workgroups=workgroups)
        h.upload_dense(pr.bed, lut)
        h.set_precision(precision)
        h.sweep(order, u, z)
        out.append(h.get_state())
        h.close()
    before.close()
    assert np.count_nonzero(out[0]["beta"]) > 0
    for st in out[1:]:
        for k in ("eps", "beta", "comp", "acum"):
            assert np.array_equal(out[0][k], st[k]), k
