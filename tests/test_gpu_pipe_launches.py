"""Chains of the pipelined sweep that take several launches: equal, bit for bit, to the same chain one iteration per
call. (An iteration's Gram entries are the same whether its blocks are split over the individuals or not: the split
parts are integer sums.)"""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
import test_zz_no_alloc as na
from _data import make_problem

pytestmark = pytest.mark.gpu

DENSE, RAGGED, EIGEN = brr.LAYOUT_DENSE_2BIT, brr.LAYOUT_RAGGED, brr.LAYOUT_EIGEN_SPARSE
S4 = [0.01, 0.001, 0.0001]


def context(pr, layout, precision, groups, fixed):
    h = brr.HipSweep(pr.n, pr.m, 4, groups, layout, ragged_storage=brr.STORAGE_CODES)
    if layout == DENSE:
        h.upload_dense(pr.bed, pr.lut)
    else:
        h.upload_ragged(pr.ragged if layout == RAGGED else brr.build_eigen(pr.bed, pr.n))
    h.set_model(np.tile(np.array(S4), (groups, 1)))
    if groups > 1:
        h.set_groups((np.arange(pr.m) % groups).astype(np.int32))
    h.set_precision(precision, 1024)
    if fixed:
        h.set_fixed(np.random.default_rng(5).normal(size=(pr.n, fixed)).astype(np.float32))
    eps, sc = brr.bayesr_init(pr.y, groups, 4, 9)
    h.set_state(eps, np.zeros(pr.m), np.zeros(pr.m, np.int32))
    h.set_scalars(sc["mu"], sc["sigmaE"], sc["epsilon_sum"], sc["sigmaG"], sc["pi"])
    return h


# (N, M, iterations): the remaining iterations of a chain's last launch hold fewer blocks than a split one would
# (1,000 x 67: 65 iterations fill a launch; 3,000 x 23: 21 do)
@pytest.mark.parametrize("n,m,iters", [(2500, 1000, 67), (2500, 3000, 23)])
@pytest.mark.parametrize("layout,precision,groups,fixed,miss", [
    (DENSE, brr.PRECISION_FP64, 1, 0, 0.0), (DENSE, brr.PRECISION_FP64, 1, 0, 0.02),
    (RAGGED, brr.PRECISION_FP32_REFRESH, 3, 2, 0.01), (EIGEN, brr.PRECISION_FP64, 2, 0, 0.01)],
    ids=["dense", "dense-missing", "ragged-fp32-groups-fixed", "eigen-groups"])
def test_chain_equals_single_iterations(gpu_lib, n, m, iters, layout, precision, groups, fixed, miss):
    pr = make_problem(n, m, seed=m + iters, causal_frac=0.01, miss=miss)
    order = np.arange(m, dtype=np.uint32)
    orders = np.stack([brr.shuffle(3, it, 0, order).copy() for it in range(iters)])
    out = []
    for step in (iters, 1):
        h = context(pr, layout, precision, groups, fixed)
        hist = np.concatenate([h.run_chain(9, 0, it, orders[it:it + step]) for it in range(0, iters, step)])
        out.append((hist, h.get_state(), h.get_scalars()))
        h.close()
    assert np.array_equal(out[0][0], out[1][0])
    for k in ("eps", "beta", "comp", "acum"):
        assert np.array_equal(out[0][1][k], out[1][1][k]), k
    for k in ("v", "betasqn", "sigmaG", "pi"):
        assert np.array_equal(out[0][2][k], out[1][2][k]), k


def test_reload_that_gains_missing_calls(gpu_lib):
    """A context loaded without missing calls, then with some: more products a block, in a chain of several launches
    and in single iterations whose blocks are split."""
    n, m, iters = 2500, 1000, 67
    a, b = (make_problem(n, m, seed=71, causal_frac=0.01, miss=x) for x in (0.0, 0.02))
    order = np.arange(m, dtype=np.uint32)
    orders = np.stack([brr.shuffle(3, it, 0, order).copy() for it in range(iters)])
    fresh = context(b, DENSE, brr.PRECISION_FP64, 1, 0)
    h = context(a, DENSE, brr.PRECISION_FP64, 1, 0)
    h.run_chain(9, 0, 0, orders[:3])
    h.upload_dense(b.bed, b.lut)
    eps, sc = brr.bayesr_init(b.y, 1, 4, 9)
    h.set_state(eps, np.zeros(m), np.zeros(m, np.int32))
    h.set_scalars(sc["mu"], sc["sigmaE"], sc["epsilon_sum"], sc["sigmaG"], sc["pi"])
    want = np.concatenate([fresh.run_chain(9, 0, it, orders[it:it + 1]) for it in range(iters)])
    got = h.run_chain(9, 0, 0, orders)
    assert np.array_equal(got, want)
    for k, x in fresh.get_state().items():
        assert np.array_equal(h.get_state()[k], x), k
    fresh.close()
    h.close()


def rel(a, b):
    a, b = np.asarray(a, float), np.asarray(b, float)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


# more markers than the Gram workspace has rows (262,144): each iteration in two launches. Sweeps against the oracle and
# against the sweep that allocates nothing, then whole iterations against the oracle's. (262,144 + 65: the parts end inside
# no block and the last one is short of a block)
@pytest.mark.parametrize("layout,groups", [(DENSE, 1), (RAGGED, 2)], ids=["dense", "ragged-groups"])
def test_iteration_in_parts(gpu_lib, layout, groups):
    n, m = 64, 262144 + 65
    pr = make_problem(n, m, seed=7, causal_frac=0.0001, maf=(0.3, 0.5))
    S = np.tile(np.array(S4), (groups, 1))
    group = (np.arange(m) % groups).astype(np.int32) if groups > 1 else None
    kw = dict(bed=pr.bed, lut=pr.lut) if layout == DENSE else dict(ragged=pr.ragged)
    o = orc.OracleProblem(n, m, layout, 4, groups, S, group=group, **kw)
    o.init(pr.y, 9)
    a, b = (context(pr, layout, brr.PRECISION_FP64, groups, 0) for _ in range(2))
    order = np.arange(m, dtype=np.uint32)
    for it in range(2):
        brr.shuffle(5, it, 0, order)
        u, z = brr.marker_uz(5, it, 0, m)
        o.sweep(order, u, z, trace=False)
        a.sweep(order, u, z)
        assert na.noalloc(b, order, u, z) == 0, brr.lib().brr_hip_last_error(b.ctx)
        sa, sb, ca, cb = a.get_state(), b.get_state(), a.get_scalars(), b.get_scalars()
        assert np.count_nonzero(o.beta) > 100
        assert np.array_equal(sa["comp"], o.comp) and np.array_equal(ca["v"].reshape(-1), o.v), it
        for k, want in (("beta", o.beta), ("acum", o.acum), ("eps", o.eps)):
            assert rel(sa[k], want) <= 1e-9, (it, k)
        assert rel(ca["betasqn"], o.betasqn) <= 1e-9, it
        for k in sa:
            assert np.array_equal(sa[k], sb[k]), (it, k)
        assert np.array_equal(ca["v"], cb["v"]) and np.array_equal(ca["betasqn"], cb["betasqn"])
        assert a.stats()["rounds"] == 4097 + 1 and a.stats()["changes"] == b.stats()["changes"]
    a.close()
    b.close()
    iters = 2
    o = orc.OracleProblem(n, m, layout, 4, groups, S, group=group, **kw)
    hist_o, _ = o.run_gibbs(pr.y, 9, iters)
    cur = np.arange(m, dtype=np.uint32)
    orders = np.stack([brr.shuffle(9, it, 0, cur).copy() for it in range(iters)])
    h = context(pr, layout, brr.PRECISION_FP64, groups, 0)
    hist = h.run_chain(9, 0, 0, orders)
    assert np.array_equal(hist[:, 2], hist_o[:, 2]) and rel(hist, hist_o) <= 1e-8
    st = h.get_state()
    assert np.array_equal(st["comp"], o.comp) and rel(st["beta"], o.beta) <= 1e-8 and rel(st["eps"], o.eps) <= 1e-8
    h.close()
