"""A residual so large that num^2 is past the largest double: every component's guard fires (BayesRBase.cpp:335), so
acum is 0, no component is drawn and beta stays, as in the oracle. Every sweep kernel."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
from _data import make_problem

pytestmark = pytest.mark.gpu

S = [0.1, 0.01, 0.001, 0.0001]


@pytest.mark.parametrize("K", [2, 3, 4, 5])
@pytest.mark.parametrize("kind", ["dense", "ragged", "lists", "batch", "block1"])
def test_guard_of_an_infinite_square(gpu_lib, K, kind):
    pr = make_problem(300, 20, seed=3)
    dense = kind in ("dense", "batch", "block1")
    S_ = np.array(S[: K - 1])
    kw = dict(bed=pr.bed, lut=pr.lut) if dense else dict(ragged=pr.ragged)
    o = orc.OracleProblem(pr.n, pr.m, orc.DENSE if dense else orc.RAGGED, K, 1, S_, **kw)
    o.init(pr.y, 3)
    o.eps[:] *= 1e160
    T = 3 if kind == "batch" else 0
    h = brr.HipSweep(pr.n, pr.m, K, 1, brr.LAYOUT_DENSE_2BIT if dense else brr.LAYOUT_RAGGED, traits=T,
                     block_markers=1 if kind == "block1" else 0,
                     ragged_storage=brr.STORAGE_LISTS if kind == "lists" else brr.STORAGE_CODES)
    h.upload_dense(pr.bed, pr.lut) if dense else h.upload_ragged(pr.ragged)
    h.set_model(S_)
    wide = (lambda a: np.stack([a] * T, axis=1)) if T else (lambda a: a)
    h.set_state(wide(o.eps), wide(o.beta), wide(o.comp))
    for t in range(max(T, 1)):
        h.set_scalars(o.mu, o.sigmaE, o.epsSum, o.sigmaG, o.pi, trait=t)
    order = np.arange(pr.m, dtype=np.uint32)
    u, z = brr.marker_uz(3, 0, 0, pr.m)
    o.sweep(order, u, z, trace=False)
    h.sweep(order, wide(u), wide(z))
    st = h.get_state()
    assert not o.acum.any() and not o.beta.any()
    for k, want in (("acum", o.acum), ("beta", o.beta), ("comp", o.comp), ("eps", o.eps)):
        assert np.array_equal(st[k], wide(want)), k
    h.close()
