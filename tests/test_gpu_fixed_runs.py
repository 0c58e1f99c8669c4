"""Chains with fixed effects on the pipelined sweep, all its kernels: layouts, precisions, one and two runs of a lane,
and iterations in parts.

Bars as the chain tests without fixed effects: FP64 within 1e-8 of the oracle's chain, FP32_REFRESH within 1e-5 (beta
2e-6), components and m0 identical. In parts (too many markers for a chain that no FP32 choice flips) the residual is
y_std - mu - X beta - F gamma within 1e-9, as FP32_REFRESH holds it in FP64."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr
import _oracle as orc
from _data import make_problem

pytestmark = pytest.mark.gpu

S = np.array([0.01, 0.001, 0.0001])
LAYOUTS = {"dense": orc.DENSE, "ragged": orc.RAGGED, "eigen": orc.EIGEN}
SEED = 20261204


def rel(a, b):
    return np.max(np.abs(np.asarray(a) - np.asarray(b))) / max(1.0, np.max(np.abs(b)))


def problem(n, m, fixed, **kw):
    pr = make_problem(n, m, seed=n + m, **kw)
    X = np.random.default_rng(fixed).normal(size=(n, fixed)).astype(np.float32)
    return pr, X, pr.y + X.astype(np.float64) @ np.linspace(0.5, -0.3, fixed)


def chain(pr, X, y, layout, precision, workgroups, iters):
    arena = pr.ragged if layout == orc.RAGGED else brr.build_eigen(pr.bed, pr.n) if layout == orc.EIGEN else None
    h = brr.HipSweep(pr.n, pr.m, 4, 1, layout, workgroups=workgroups, ragged_storage=brr.STORAGE_CODES)
    h.upload_dense(pr.bed, pr.lut) if layout == orc.DENSE else h.upload_ragged(arena)
    h.set_model(S)
    h.set_precision(precision, 1024)
    h.set_fixed(X)
    eps, sc = brr.bayesr_init(y, 1, 4, SEED)
    h.set_state(eps, np.zeros(pr.m), np.zeros(pr.m, np.int32))
    h.set_scalars(sc["mu"], sc["sigmaE"], sc["epsilon_sum"], sc["sigmaG"], sc["pi"])
    cur = np.arange(pr.m, dtype=np.uint32)
    orders = np.stack([brr.shuffle(SEED, it, 0, cur).copy() for it in range(iters)])
    hist = h.run_chain(SEED, 0, 0, orders)
    out = hist, h.get_state(), h.get_fixed_state(), h.get_scalars()
    h.close()
    return out, eps + sc["mu"], arena


@pytest.mark.parametrize("fixed", [1, 4])
@pytest.mark.parametrize("workgroups", [2, 4], ids=["two-runs", "one-run"])      # 1,900: slices of 950 and 475
@pytest.mark.parametrize("precision", [brr.PRECISION_FP64, brr.PRECISION_FP32_REFRESH], ids=["fp64", "fp32"])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_chain_against_oracle(gpu_lib, layout, precision, workgroups, fixed):
    iters = 4
    pr, X, y = problem(1900, 150, fixed, causal_frac=0.05, miss=0.02)
    (hist, st, fx, sc), _, arena = chain(pr, X, y, LAYOUTS[layout], precision, workgroups, iters)
    kw = dict(bed=pr.bed, lut=pr.lut) if arena is None else dict(ragged=arena)
    o = orc.OracleProblem(pr.n, pr.m, LAYOUTS[layout], 4, 1, S, **kw)
    o.set_fixed(X)
    want, _ = o.run_gibbs_fixed(y, SEED, iters)
    bar, beta_bar = (1e-8, 1e-8) if precision == brr.PRECISION_FP64 else (1e-5, 2e-6)
    assert np.array_equal(hist[:, 2], want[:, 2]) and np.array_equal(st["comp"], o.comp)
    assert np.array_equal(fx["order"], o.forder)
    assert np.max(np.abs(hist - want) / np.maximum(np.abs(want), 1.0)) <= bar
    assert rel(st["eps"], o.eps) <= bar and rel(fx["gamma"], o.gamma) <= bar
    assert rel(st["beta"], o.beta) <= beta_bar


@pytest.mark.parametrize("layout", LAYOUTS)
def test_parts_keep_the_residual(gpu_lib, layout):
    pr, X, y = problem(64, 262_144 + 65, 3, causal_frac=0.0001, maf=(0.3, 0.5))
    (_, st, fx, sc), y_std, _ = chain(pr, X, y, LAYOUTS[layout], brr.PRECISION_FP32_REFRESH, 0, 2)
    at = np.flatnonzero(st["beta"])
    assert at.size > 0 and np.all(fx["gamma"] != 0)
    bits = np.unpackbits(pr.bed[at][..., None], axis=-1, bitorder="little").reshape(at.size, -1)
    dosage = np.array([2, 3, 1, 0])[(bits[:, 0::2] | (bits[:, 1::2] << 1))[:, :pr.n]]
    xb = st["beta"][at] @ np.take_along_axis(pr.lut[at], dosage, axis=1)
    assert rel(st["eps"], y_std - sc["mu"] - xb - X.astype(np.float64) @ fx["gamma"]) <= 1e-9
