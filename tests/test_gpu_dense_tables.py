"""Dense sweeps over tables that are not a builder's: any four values per column, whatever code holds which. The Gram
entries of the pipelined sweep follow the table as the dots and the residual update do.

Bars as in the other sweep tests: beta, acum and epsilon within 1e-9 of the FP64 oracle, components and counts identical."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
from _data import make_problem, spec_dosage

pytestmark = pytest.mark.gpu

S4 = np.array([0.01, 0.001, 0.0001])
BAR = 1e-9


def rel(a, b):
    a, b = np.asarray(a, float), np.asarray(b, float)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


def ppbed(pr):
    """The problem's columns as a preprocessed file read back: codes numbered by first appearance in each column."""
    x = np.ascontiguousarray(pr.x_dense().T)
    size = x.shape[1] * 8
    index = np.array([[j * size, size, size] for j in range(pr.m)], dtype=np.uint64)
    bed, lut = brr.read_ppbed(x.tobytes(), index, pr.n)
    steps = np.abs(2 * lut[:, 1] - lut[:, 0] - lut[:, 2]) <= 1e-9
    assert not np.all(steps)              # (tables that are linear in the code by chance only)
    return bed, lut


def free_tables(pr, seed, three=False):
    """Random values per code, standardised over the individuals; three: the missing call shares dosage 0's value."""
    rng = np.random.default_rng(seed)
    lut = rng.normal(size=(pr.m, 4))
    if three:
        lut[:, 3] = lut[:, 0]
    d = spec_dosage(pr.bed, pr.n)
    x = np.take_along_axis(lut, np.where(d < 0, 3, d), axis=1)
    return pr.bed, (lut - x.mean(axis=1)[:, None]) / x.std(axis=1, ddof=1)[:, None]


def two_dosages(pr, seed):
    """Columns in which one dosage does not occur, beside some with one value only; a builder's tables."""
    d = np.abs(spec_dosage(pr.bed, pr.n))
    for j in range(pr.m):
        a, b = [(2, 1), (0, 1), (1, 2)][j % 3]
        d[j][d[j] == a] = b
    codes = np.zeros((pr.m, 4 * pr.bed.shape[1]), dtype=np.uint8)
    codes[:, :pr.n] = np.array([3, 2, 0], dtype=np.uint8)[d]
    q = codes.reshape(pr.m, -1, 4)
    bed = q[..., 0] | q[..., 1] << 2 | q[..., 2] << 4 | q[..., 3] << 6
    lut = brr.build_dense(bed, pr.n)
    lut[0] = 0.0
    lut[~np.isfinite(lut).all(axis=1)] = 0.0      # (columns of one value have no standard deviation)
    return bed, lut


def pair(pr, bed, lut, **kw):
    o = orc.OracleProblem(pr.n, pr.m, orc.DENSE, 4, 1, S4, bed=bed, lut=lut)
    o.init(pr.y, 11)
    o.beta[:] = np.random.default_rng(3).normal(0.0, 0.02, pr.m)      # in the model, so that every sweep changes many
    o.comp[:] = 1 + np.arange(pr.m) % 3
    o.pi[:] = [0.4, 0.2, 0.2, 0.2]
    h = brr.HipSweep(pr.n, pr.m, 4, 1, brr.LAYOUT_DENSE_2BIT, **kw)
    h.upload_dense(bed, lut)
    h.set_model(S4)
    h.set_state(o.eps, o.beta, o.comp)
    h.set_scalars(o.mu, o.sigmaE, o.epsSum, o.sigmaG, o.pi)
    return o, h


# (N, M, block): Gram launches split over the individuals and not, blocks with a next one and without
@pytest.mark.parametrize("n,m,block", [(700, 61, 0), (1025, 129, 33), (5001, 200, 0), (400, 8300, 0)])
@pytest.mark.parametrize("tables", ["ppbed", "ppbed-missing", "three", "four", "two"])
def test_sweep_follows_the_table(gpu_lib, n, m, block, tables):
    miss = 0.0 if tables == "ppbed" else 0.03
    pr = make_problem(n, m, seed=n + m, causal_frac=0.05, maf=(0.1, 0.5), miss=miss)
    bed, lut = (ppbed(pr) if tables.startswith("ppbed") else two_dosages(pr, n) if tables == "two" else
                free_tables(pr, n, tables == "three"))
    o, h = pair(pr, bed, lut, block_markers=block)
    order = np.arange(m, dtype=np.uint32)
    for it in range(2):
        brr.shuffle(5, it, 0, order)
        u, z = brr.marker_uz(5, it, 0, m)
        o.sweep(order, u, z, trace=False)
        h.sweep(order, u, z)
        st = h.get_state()
        assert np.array_equal(st["comp"], o.comp), it
        for k, want in (("beta", o.beta), ("acum", o.acum), ("eps", o.eps)):
            assert rel(st[k], want) <= BAR, (it, k)
    h.close()


# a cohort with such tables beside one with a builder's
def test_cohorts_follow_the_table(gpu_lib):
    prs = [make_problem(1500, 150, seed=81, causal_frac=0.1, miss=0.02), make_problem(900, 300, seed=82, causal_frac=0.1)]
    tabs = [free_tables(prs[0], 5), ppbed(prs[1])]
    iters = 3
    orders = []
    for q, pr in enumerate(prs):
        cur = np.arange(pr.m, dtype=np.uint32)
        orders.append(np.stack([brr.shuffle(7, it, q, cur).copy() for it in range(iters)]))
    hs, want = [], []
    for q, (pr, (bed, lut)) in enumerate(zip(prs, tabs)):
        o = orc.OracleProblem(pr.n, pr.m, orc.DENSE, 4, 1, S4, bed=bed, lut=lut)
        want.append((o, o.run_gibbs(pr.y, 7, iters, chain=q)[0]))
        h = brr.HipSweep(pr.n, pr.m, 4, 1, brr.LAYOUT_DENSE_2BIT)
        h.upload_dense(bed, lut)
        h.set_model(S4)
        eps, sc = brr.bayesr_init(pr.y, 1, 4, 7, chain=q)
        h.set_state(eps, np.zeros(pr.m), np.zeros(pr.m, np.int32))
        h.set_scalars(sc["mu"], sc["sigmaE"], sc["epsilon_sum"], sc["sigmaG"], sc["pi"])
        hs.append(h)
    hists, _ = brr.run_cohorts(hs, 7, 0, orders, chains=[0, 1])
    for q, (h, (o, hist)) in enumerate(zip(hs, want)):
        st = h.get_state()
        assert np.array_equal(hists[q][:, 2], hist[:, 2]) and np.array_equal(st["comp"], o.comp), q
        assert rel(hists[q], hist) <= 1e-8 and rel(st["beta"], o.beta) <= 1e-8 and rel(st["eps"], o.eps) <= 1e-8, q
        h.close()


def test_values_of_codes_that_do_not_occur(gpu_lib):
    """Without missing calls the table's last value plays no part, whatever it holds."""
    pr = make_problem(1000, 130, seed=91, causal_frac=0.1)
    out = []
    for last in (0.0, np.nan, np.inf):
        lut = pr.lut.copy()
        lut[:, 3] = last
        o, h = pair(pr, pr.bed, lut)
        order = brr.shuffle(5, 0, 0, np.arange(pr.m, dtype=np.uint32))
        h.sweep(order, *brr.marker_uz(5, 0, 0, pr.m))
        out.append(h.get_state())
        h.close()
    assert len(np.unique(out[0]["comp"])) > 1
    for st in out[1:]:
        for k in ("eps", "beta", "comp", "acum"):
            assert np.array_equal(out[0][k], st[k]), k
