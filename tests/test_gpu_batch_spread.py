"""Batched sweeps whose traits are not a multiple of what a wave decides (a quarter of them) or of a matrix-core
tile (16): decisions and residual update then belong to different waves."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
import test_gpu_batch as tb
from _data import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [2, 4, 5, 15, 16, 17, 33, 48, 63])
def test_traits_spread_over_waves(gpu_lib, T):
    pr = make_problem(700, 70, seed=400 + T, h2=0.5, causal_frac=0.1)
    seed = 41
    os_ = tb.oracle_traits(pr, orc.DENSE, tb.phenotypes(pr, T, seed=T), seed)
    h = tb.device_traits(pr, orc.DENSE, os_, workgroups=3 if T % 2 else 0)
    order = np.arange(pr.m, dtype=np.uint32)
    for it in range(2):
        brr.shuffle(seed, it, 0, order)
        uz = [brr.marker_uz(seed, it, t, pr.m) for t in range(T)]
        for t, o in enumerate(os_):
            o.sweep(order, *uz[t], trace=False)
        h.sweep(order, np.stack([a for a, _ in uz], axis=1), np.stack([b for _, b in uz], axis=1))
        tb.compare(os_, h, orc.DENSE, f"iteration {it}")
    h.close()
