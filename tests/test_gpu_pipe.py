"""The pipelined sweep and its Gram entries at the edges of what they take, against the FP64 oracle.

A sweep's beta, acum and epsilon agree with the oracle to the reduction-order bar of the other sweep tests (1e-9
relative; a Gram entry carries roundings of about 1e-16 N, which a change of beta scales down again), epsilonSum to
1e-9 of its N terms; components and counts are identical.
"""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
from _data import make_problem

pytestmark = pytest.mark.gpu

S_K = {2: [0.01], 3: [0.01, 0.001], 4: [0.01, 0.001, 0.0001], 5: [0.1, 0.01, 0.001, 0.0001],
       8: [0.1, 0.03, 0.01, 0.003, 0.001, 0.0003, 0.0001]}
BAR = 1e-9


def rel(a, b):
    a, b = np.asarray(a, float), np.asarray(b, float)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


def eigen_arena(pr):
    return brr.build_eigen(pr.bed, pr.n)


def pair(pr, layout, K=4, groups=1, workgroups=0, block=0):
    S = np.tile(np.array(S_K[K]), (groups, 1))
    group = (np.arange(pr.m) % groups).astype(np.int32) if groups > 1 else None
    arena = eigen_arena(pr) if layout == orc.EIGEN else pr.ragged
    kw = dict(bed=pr.bed, lut=pr.lut) if layout == orc.DENSE else dict(ragged=arena)
    o = orc.OracleProblem(pr.n, pr.m, layout, K, groups, S, group=group, **kw)
    o.init(pr.y, 11)
    h = brr.HipSweep(pr.n, pr.m, K, groups, layout, workgroups=workgroups, block_markers=block,
                     ragged_storage=brr.STORAGE_CODES)
    if layout == orc.DENSE:
        h.upload_dense(pr.bed, pr.lut)
    else:
        h.upload_ragged(arena)
    h.set_model(S)
    if group is not None:
        h.set_groups(group)
    push(o, h)
    return o, h


def push(o, h):
    h.set_state(o.eps, o.beta, o.comp)
    h.set_scalars(o.mu, o.sigmaE, o.epsSum, o.sigmaG, o.pi)


def sweeps(o, h, layout, count=2, seed=5):
    order = np.arange(h.m, dtype=np.uint32)
    for it in range(count):
        brr.shuffle(seed, it, 0, order)
        u, z = brr.marker_uz(seed, it, 0, h.m)
        o.sweep(order, u, z, trace=False)
        h.sweep(order, u, z)
        st, sc = h.get_state(), h.get_scalars()
        assert np.array_equal(st["comp"], o.comp), it
        assert np.array_equal(sc["v"].reshape(-1), o.v), it
        for k, want in (("beta", o.beta), ("acum", o.acum), ("eps", o.eps)):
            assert rel(st[k], want) <= BAR, (it, k)
        assert rel(sc["betasqn"], o.betasqn) <= BAR
        if layout != orc.DENSE:
            assert abs(sc["epsilon_sum"] - o.epsSum) <= BAR * h.n
        assert h.stats()["rounds"] == -(-h.m // h.stats()["block_markers"])   # one exchange per block


# workgroups that sum all partials themselves (<= 16), reduce four or two slots or one at a time, and the
# borders between them
@pytest.mark.parametrize("workgroups", [1, 2, 16, 17, 31, 33, 63, 64, 65, 130])
def test_exchange_variants(gpu_lib, workgroups):
    pr = make_problem(16 * workgroups + 5 if workgroups > 1 else 301, 150, seed=300 + workgroups, causal_frac=0.2)
    o, h = pair(pr, orc.RAGGED, workgroups=workgroups)
    sweeps(o, h, orc.RAGGED)
    h.close()


# blocks that are empty, partial and full, one and two lane runs, individuals at the edges of a staged chunk
@pytest.mark.parametrize("layout", [orc.DENSE, orc.RAGGED, orc.EIGEN], ids=["dense", "ragged", "eigen"])
@pytest.mark.parametrize("n,m,block,workgroups", [(64, 1, 0, 0), (65, 2, 0, 0), (1023, 64, 0, 1), (1024, 65, 0, 1),
                                                  (1025, 129, 0, 2), (2049, 130, 33, 3), (700, 61, 2, 0)])
@pytest.mark.parametrize("miss", [0.0, 0.03])
def test_sizes(gpu_lib, layout, n, m, block, workgroups, miss):
    pr = make_problem(n, m, seed=n + m, causal_frac=0.3, maf=(0.1, 0.5), miss=miss)
    o, h = pair(pr, layout, block=block, workgroups=workgroups)
    sweeps(o, h, layout, 3)
    h.close()


# every marker in the model: more in-model slots than Gram rows are held, changes at every slot
@pytest.mark.parametrize("layout", [orc.DENSE, orc.RAGGED, orc.EIGEN], ids=["dense", "ragged", "eigen"])
@pytest.mark.parametrize("workgroups", [0, 1])
@pytest.mark.parametrize("K,groups", [(2, 1), (3, 2), (4, 1), (5, 3), (8, 1)])
def test_all_in_model(gpu_lib, layout, workgroups, K, groups):
    pr = make_problem(900, 200, seed=17 * K + groups, causal_frac=0.9, miss=0.01)
    o, h = pair(pr, layout, K=K, groups=groups, workgroups=workgroups)
    rng = np.random.default_rng(K)
    o.beta[:] = rng.normal(0.0, 0.02, pr.m)
    o.comp[:] = 1 + np.arange(pr.m) % (K - 1)
    o.pi[:] = np.tile([0.02] + [0.98 / (K - 1)] * (K - 1), groups)
    push(o, h)
    sweeps(o, h, layout, 3)
    h.close()


# log-likelihood gaps past 350 and past the 700 guard beside small ones, and components of prior probability 0
@pytest.mark.parametrize("layout", [orc.DENSE, orc.RAGGED], ids=["dense", "ragged"])
@pytest.mark.parametrize("K,pi", [(4, None), (4, [0.0, 0.5, 0.3, 0.2]), (4, [0.5, 0.0, 0.3, 0.2]), (3, [0.0, 0.6, 0.4]),
                                  (2, [0.3, 0.7]), (5, [0.4, 0.2, 0.0, 0.2, 0.2])])
def test_far_components(gpu_lib, layout, K, pi):
    pr = make_problem(4000, 140, seed=77, h2=0.9, causal_frac=0.02)
    o, h = pair(pr, layout, K=K)
    o.state.sigmaE = 0.02          # large effects against a small residual variance
    if pi is not None:
        o.pi[:] = pi
    push(o, h)
    sweeps(o, h, layout, 3)
    h.close()


def test_chain_over_several_launches(gpu_lib):
    """A chain whose Gram rows take several launches (65,536 rows each) equals the same chain one iteration per call."""
    pr = make_problem(400, 9000, seed=5, causal_frac=0.01)
    iters = 9                      # 7 iterations fill a launch
    orders = np.stack([brr.shuffle(3, it, 0, np.arange(pr.m, dtype=np.uint32)) for it in range(iters)])
    out = []
    for step in (iters, 1):
        o, h = pair(pr, orc.DENSE)
        hist = np.concatenate([h.run_chain(9, 0, it, orders[it:it + step]) for it in range(0, iters, step)])
        out.append((hist, h.get_state()))
        h.close()
    assert np.array_equal(out[0][0], out[1][0])
    for k in ("eps", "beta", "comp", "acum"):
        assert np.array_equal(out[0][1][k], out[1][1][k]), k
