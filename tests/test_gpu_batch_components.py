"""Batched draws over every component count: the straight-line draw pads its constants beyond the last component, which
must add nothing, guard nothing and never be drawn -- beside log-likelihood gaps past 350 and past the 700 guard, and
components of prior probability 0."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
import test_gpu_batch as tb
from _data import make_problem

pytestmark = pytest.mark.gpu

S8 = [0.1, 0.03, 0.01, 0.003, 0.001, 0.0003, 0.0001]


@pytest.mark.parametrize("layout", [orc.DENSE, orc.RAGGED], ids=["dense", "ragged"])
@pytest.mark.parametrize("K", [2, 3, 4, 5, 6, 7, 8])
def test_component_counts_with_far_gaps(gpu_lib, K, layout):
    pr = make_problem(3000, 100, seed=50 + K, h2=0.9, causal_frac=0.03)
    T = 7
    ys = tb.phenotypes(pr, T, seed=K)
    S = np.array(S8[: K - 1])
    kw = dict(bed=pr.bed, lut=pr.lut) if layout == orc.DENSE else dict(ragged=pr.ragged)
    os_ = []
    for t, y in enumerate(ys):
        o = orc.OracleProblem(pr.n, pr.m, layout, K, 1, S, **kw)
        o.init(y, 31, chain=t)
        if t % 2:
            o.state.sigmaE = 0.02          # large effects against a small residual variance
        pi = np.full(K, 1.0)
        if t >= 2 and K > 2:
            pi[t % K] = 0.0                # a component that is never drawn, the zero component among them
        o.pi[:] = pi / pi.sum()
        os_.append(o)
    code = brr.LAYOUT_DENSE_2BIT if layout == orc.DENSE else brr.LAYOUT_RAGGED
    h = brr.HipSweep(pr.n, pr.m, K, 1, code, traits=T)
    h.upload_dense(pr.bed, pr.lut) if layout == orc.DENSE else h.upload_ragged(pr.ragged)
    h.set_model(S)
    h.set_state(np.stack([o.eps for o in os_], axis=1), np.zeros((pr.m, T)), np.zeros((pr.m, T), np.int32))
    for t, o in enumerate(os_):
        h.set_scalars(o.mu, o.sigmaE, o.epsSum, o.sigmaG, o.pi, trait=t)
    order = np.arange(pr.m, dtype=np.uint32)
    for it in range(3):
        brr.shuffle(31, it, 0, order)
        uz = [brr.marker_uz(31, it, t, pr.m) for t in range(T)]
        for o, (u, z) in zip(os_, uz):
            o.sweep(order, u, z, trace=False)
        h.sweep(order, np.stack([a for a, _ in uz], axis=1), np.stack([b for _, b in uz], axis=1))
        tb.compare(os_, h, layout, f"iteration {it}")
    h.close()
