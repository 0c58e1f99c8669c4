"""The work that programs have this package do, as cases that a timing harness runs.

A case is one call of the public entry points on data of a stated size:

  exec     one AnalysisGraph::exec of a host-driven runGibbs: the host hands in its residual,
           betas and scalars, the sweep runs over a marker order with the host's u and z, and the
           updated state comes back (the HipSweepGraph binding).
  chain    a resident chain run in chunks that end on a kept sample: run_chain, then get_state.
  batch    the same two ways of use with T traits over one genotype matrix.
  bayesw   a resident BayesW chain in chunks.
  cohorts  chains of uneven cohorts side by side, then every cohort's state.
  decode   a whole .bed file image decoded into a context, and its per-marker tables.

Genotypes are Hardy-Weinberg draws with MAF ~ U(maf_lo, maf_hi), a set of causal markers with normal
effects and normal (BayesW: log-Weibull, 10% censored) noise. Chains start from the simulated truth,
so that the work of an iteration is the work late in a chain; only `start = init` starts from
BayesRBase::init with every marker out of the model.
"""
import math

import numpy as np
import torch

import bayesrrcmd_amd as brr

S_OF_K = {2: (0.001,), 3: (0.001, 0.0001), 4: (0.01, 0.001, 0.0001), 5: (0.1, 0.01, 0.001, 0.0001),
          8: (0.03, 0.01, 0.003, 0.001, 0.0003, 0.0001, 0.00003)}
LAYOUTS = {"dense": brr.LAYOUT_DENSE_2BIT, "ragged": brr.LAYOUT_RAGGED, "lists": brr.LAYOUT_RAGGED,
           "eigen": brr.LAYOUT_EIGEN_SPARSE}
H2 = 0.4


def _case(kind, n, m, **kw):
    c = {"kind": kind, "n": n, "m": m, "layout": "dense", "precision": "fp64", "maf_lo": 0.01, "maf_hi": 0.5,
         "miss": 0.0, "K": 4, "groups": 1, "causal": 0.005, "traits": 0, "window": 0, "iterations": 1, "start": "truth",
         "cohorts": 0, "host": kind == "exec"}
    c.update(kw)
    return c


def listed():
    return [
        # a test-sized data set through the host-driven binding: launch and copy latency
        _case("exec", 503, 200, name="exec small dense", causal=0.05),
        # rare variants, held as index lists because those are smaller; groups and missing calls
        _case("exec", 30000, 4001, name="exec rare lists", layout="lists", maf_lo=0.002, maf_hi=0.02, miss=0.0005,
              groups=3),
        # the plain chain at the headline's N and precision (ragged input, FP32 residual, FP64 refresh)
        _case("chain", 100000, 20000, name="chain ragged 100k fp32", layout="ragged", precision="fp32", maf_lo=0.005,
              iterations=2),
        # the default precision at a ragged size between the tuned ones
        _case("chain", 60013, 8009, name="chain dense 60k fp64", miss=0.002, iterations=3),
        # a new analysis of the small dense configuration: burn-in, where half the markers change
        _case("chain", 5000, 10000, name="chain small from init", causal=0.01, iterations=2, start="init"),
        # 64 phenotypes over one matrix
        _case("batch", 50000, 4000, name="batch 64 traits 50k fp32", precision="fp32", traits=64, iterations=4),
        _case("batch", 100000, 2400, name="batch 64 traits 100k fp32", precision="fp32", traits=64, iterations=3,
              maf_lo=0.005),
        # a few phenotypes of a small cohort, FP64, host-driven
        _case("batch", 7003, 1501, name="batch 20 traits 7k fp64", layout="ragged", traits=20, miss=0.01, causal=0.01,
              host=True),
        # survival model, the large ragged configuration's N and a small dense one
        _case("bayesw", 100000, 6000, name="bayesw ragged 100k", layout="ragged", maf_lo=0.005, iterations=3),
        _case("bayesw", 3001, 701, name="bayesw small dense", causal=0.02, maf_lo=0.05, iterations=4),
        # uneven cohorts in one launch
        _case("cohorts", 40000, 6000, name="cohorts 8 uneven", cohorts=8, iterations=2),
        # a .bed image to device-resident markers
        _case("decode", 100000, 8000, name="decode dense 100k", maf_lo=0.005, miss=0.005),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["exec", "exec", "chain", "chain", "batch", "batch", "bayesw", "cohorts", "decode"])
    causal = rng.choice([0.002, 0.005, 0.01])
    miss = rng.choice([0.0, 0.0, 0.002, 0.01])
    maf_lo = rng.choice([0.005, 0.01, 0.05])
    if kind in ("exec", "chain"):
        n = _logu(rng, 300, 100000)
        m = _logu(rng, 100, 8000)
        layout = rng.choice(["dense", "ragged", "ragged", "eigen"] + (["lists"] if kind == "exec" else []))
        c = _case(kind, n, m, layout=layout, causal=causal, miss=miss, maf_lo=maf_lo, K=rng.choice([3, 4, 4, 4, 5, 8]),
                  groups=rng.choice([1, 1, 1, 4]), iterations=1 if kind == "exec" else rng.choice([1, 2, 4]))
        if layout == "lists":
            c.update(n=min(n, 40000), maf_lo=0.002, maf_hi=0.02, miss=rng.choice([0.0, 0.0005]))
        elif rng.random() < 0.4:
            c["precision"] = "fp32"
        elif rng.random() < 0.2:
            c["window"] = rng.choice([7, 20, 64])
        return c
    if kind == "batch":
        n = _logu(rng, 2000, 100000)
        fp32 = n > 60000 or rng.random() < 0.6
        return _case(kind, n, _logu(rng, 200, 2400), layout=rng.choice(["dense", "dense", "ragged"]),
                     traits=rng.choice([5, 20, 33, 64]), precision="fp32" if fp32 else "fp64", causal=causal,
                     miss=miss, maf_lo=maf_lo,
                     **rng.choice([dict(iterations=1), dict(iterations=2), dict(host=True)]))
    if kind == "bayesw":
        return _case(kind, _logu(rng, 2000, 100000), _logu(rng, 200, 5000), layout=rng.choice(["dense", "ragged"]),
                     causal=rng.choice([0.005, 0.01]), miss=miss, maf_lo=max(0.01, maf_lo),
                     iterations=rng.choice([1, 2]))
    if kind == "cohorts":
        return _case(kind, _logu(rng, 5000, 40000), _logu(rng, 500, 5000), cohorts=rng.randint(2, 8), causal=causal,
                     iterations=rng.choice([1, 2]), precision=rng.choice(["fp64", "fp32"]))
    return _case(kind, _logu(rng, 500, 100000), _logu(rng, 500, 8000), layout=rng.choice(["dense", "ragged", "eigen"]),
                 miss=miss, maf_lo=maf_lo)


# ------------------------------------------------------------------ inputs --

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _codes(n, m, maf_lo, maf_hi, miss, seed):
    """(m, n) PLINK 2-bit values on the GPU: 0 = dosage 2, 1 = missing, 2 = dosage 1, 3 = dosage 0."""
    g = torch.Generator(device=_dev()).manual_seed(seed)
    out = torch.empty((m, n), dtype=torch.uint8, device=_dev())
    rows = max(1, (1 << 26) // n)
    for a in range(0, m, rows):
        b = min(m, a + rows)
        maf = torch.rand((b - a, 1), generator=g, device=_dev()) * (maf_hi - maf_lo) + maf_lo
        r = torch.rand((b - a, n), generator=g, device=_dev())
        # dosage 2 with p^2, 1 with 2 p (1 - p), the rest 0
        code = torch.full((b - a, n), 3, dtype=torch.uint8, device=_dev())
        code[r < 2 * maf - maf * maf] = 2
        code[r < maf * maf] = 0
        if miss:
            code[torch.rand((b - a, n), generator=g, device=_dev()) < miss] = 1
        # no column without a carrier
        at = torch.arange(a, b, device=_dev())
        code[at - a, at % n] = 2
        out[a:b] = code
    return out


def _packed(codes):
    """The columns' ceil(n / 4) bytes."""
    m, n = codes.shape
    cb = (n + 3) // 4
    if n % 4:
        codes = torch.nn.functional.pad(codes, (0, 4 * cb - n))
    q = codes.view(m, cb, 4)
    return q[..., 0] | (q[..., 1] << 2) | (q[..., 2] << 4) | (q[..., 3] << 6)


def _bed_image(codes):
    """A .bed file's bytes in host memory."""
    p = _packed(codes).reshape(-1)
    magic = torch.tensor([0x6C, 0x1B, 0x01], dtype=torch.uint8, device=p.device)
    return torch.cat([magic, p]).cpu().numpy()


def _mixture(K, groups):
    return np.tile(np.array(S_OF_K[K]), (groups, 1))


def _truth(c, rng, cols):
    """Simulated effects (m,) or (m, T), their components, and the pi that goes with them."""
    m = c["m"]
    S = np.array(S_OF_K[c["K"]])
    beta, comp = np.zeros((m, cols)), np.zeros((m, cols), dtype=np.int32)
    for t in range(cols):
        mc = max(1, int(round(c["causal"] * m)))
        at = rng.choice(m, mc, replace=False)
        b = rng.normal(0.0, math.sqrt(H2 / mc), mc)
        beta[at, t] = b
        # the component whose variance is nearest to the effect's
        comp[at, t] = 1 + np.argmin(np.abs(np.log(S[None, :] * H2) - np.log(b * b + 1e-12)[:, None]), axis=1)
    pi = np.full(c["K"], 2.0 * c["causal"] / (c["K"] - 1))
    pi[0] = 1.0 - pi[1:].sum()
    return beta, comp, pi


def _orders(rng, m, count):
    return np.stack([rng.permutation(m).astype(np.uint32) for _ in range(count)])


def _bayesr_inputs(c, seed):
    """Everything of a BayesR case but the genotypes, as host arrays."""
    rng = np.random.default_rng(seed + 1)
    T = max(1, c["traits"])
    beta, comp, pi = _truth(c, rng, T)
    eps = rng.normal(0.0, math.sqrt(1.0 - H2), (c["n"], T))
    x = dict(eps=eps, beta=beta, comp=comp, pi=np.tile(pi, (c["groups"], 1)), sigmaE=1.0 - H2,
             sigmaG=np.full(c["groups"], H2 / c["groups"]), S=_mixture(c["K"], c["groups"]),
             orders=_orders(rng, c["m"], c["iterations"]),
             group=rng.integers(0, c["groups"], c["m"]).astype(np.int32))
    if c["host"]:
        x["u"], x["z"] = rng.random((c["m"], T)), rng.normal(0.0, 1.0, (c["m"], T))
    if not c["traits"]:
        for k in ("eps", "beta", "comp", "u", "z"):
            if k in x:
                x[k] = np.ascontiguousarray(x[k][:, 0])
    return x


# ----------------------------------------------------------------- prepare --

def _upload(h, c, codes):
    if c["layout"] == "lists":
        h.upload_ragged(brr.build_ragged(_packed(codes).cpu().numpy(), c["n"]))
    else:
        h.load_bed(_bed_image(codes), LAYOUTS[c["layout"]])


def _sweep_context(c, x, codes):
    h = brr.HipSweep(c["n"], c["m"], c["K"], c["groups"], LAYOUTS[c["layout"]], traits=c["traits"])
    if c["precision"] == "fp32":
        h.set_precision(brr.PRECISION_FP32 if c["traits"] else brr.PRECISION_FP32_REFRESH)
    _upload(h, c, codes)
    h.set_model(x["S"])
    if c["groups"] > 1:
        h.set_groups(x["group"])
    if c["window"]:
        h.set_async(c["window"])
    _set_state(h, c, x)
    return h


def _set_state(h, c, x):
    h.set_state(x["eps"], x["beta"], x["comp"])
    if c["traits"]:
        sums = x["eps"].sum(axis=0)
        for t in range(c["traits"]):
            h.set_scalars(0.0, x["sigmaE"], sums[t], x["sigmaG"], x["pi"], trait=t)
    else:
        h.set_scalars(0.0, x["sigmaE"], x["eps"].sum(), x["sigmaG"], x["pi"])


def _from_init(c, x, codes, seed):
    """The state of BayesRBase::init for a simulated phenotype."""
    w = _weights(c, codes)[0]
    y = x["eps"].copy()
    for j in np.flatnonzero(x["beta"]):
        y += w[j][codes[j].long()].cpu().numpy() * x["beta"][j]
    eps, s = brr.bayesr_init(y.astype(np.float32).astype(np.float64), c["groups"], c["K"], seed)
    x.update(eps=eps, beta=np.zeros(c["m"]), comp=np.zeros(c["m"], dtype=np.int32), sigmaE=s["sigmaE"],
             sigmaG=s["sigmaG"], pi=s["pi"])


def _prepare_bayesw(c, seed):
    codes = _codes(c["n"], c["m"], c["maf_lo"], c["maf_hi"], c["miss"], seed)
    rng = np.random.default_rng(seed + 1)
    n, m, alpha, C = c["n"], c["m"], 3.0, np.array([0.001, 0.01, 0.1])
    mc = max(1, int(round(c["causal"] * m)))
    at = rng.choice(m, mc, replace=False)
    var_g = math.pi ** 2 / (6 * alpha ** 2)      # half the variance of log T
    sigma_b = var_g / (mc * float(C.mean()))
    comp, beta = np.zeros(m, dtype=np.int32), np.zeros(m)
    comp[at] = rng.integers(1, 4, mc)
    beta[at] = rng.normal(0.0, 1.0, mc) * np.sqrt(sigma_b * C[comp[at] - 1])
    eps = (np.log(rng.exponential(1.0, n)) + 0.5772156649015329) / alpha
    fail = np.ones(n)
    cens = rng.random(n) < 0.1
    fail[cens] = 0.0
    eps[cens] += np.log(rng.uniform(0.05, 1.0, int(cens.sum())))
    pi = np.full(4, 2.0 * c["causal"] / 3)
    pi[0] = 1.0 - pi[1:].sum()
    h = brr.HipBayesW(n, m, 4, quad_points=7)
    h.load_bed(_bed_image(codes), LAYOUTS[c["layout"]])
    h.set_model(C, fail)
    h.set_state(eps, beta, comp)
    h.set_scalars(4.0, alpha, sigma_b, float(fail.sum()), pi, np.ones(4))
    return dict(case=c, h=h, orders=_orders(rng, m, c["iterations"]), it=0, seed=seed)


def _cohorts(c):
    """The cohorts as chain cases: sizes over their logarithm down to a tenth, the same for every seed."""
    k = c["cohorts"]
    for q in range(k):
        yield dict(c, kind="chain", n=max(300, int(c["n"] * 0.1 ** (q / max(1, k - 1)))) + q,
                   m=max(100, int(c["m"] * (1.0 - 0.6 * q / k))), layout="dense" if q % 2 else "ragged")


def _prepare_cohorts(c, seed):
    hs, orders = [], []
    for q, d in enumerate(_cohorts(c)):
        x = _bayesr_inputs(d, seed + 10 * q)
        codes = _codes(d["n"], d["m"], d["maf_lo"], d["maf_hi"], d["miss"], seed + 10 * q)
        hs.append(_sweep_context(d, x, codes))
        orders.append(x["orders"])
    return dict(case=c, hs=hs, orders=orders, it=0, seed=seed)


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "bayesw":
        return _prepare_bayesw(c, seed)
    if c["kind"] == "cohorts":
        return _prepare_cohorts(c, seed)
    codes = _codes(c["n"], c["m"], c["maf_lo"], c["maf_hi"], c["miss"], seed)
    if c["kind"] == "decode":
        h = brr.HipSweep(c["n"], c["m"], c["K"], 1, LAYOUTS[c["layout"]])
        return dict(case=c, h=h, image=_bed_image(codes))
    x = _bayesr_inputs(c, seed)
    if c["start"] == "init":
        _from_init(c, x, codes, seed)
    return dict(case=c, h=_sweep_context(c, x, codes), x=x, it=0, seed=seed)


# --------------------------------------------------------------------- run --

def _scalars(h, c):
    if not c["traits"]:
        s = h.get_scalars()
        return {k: s[k] for k in ("mu", "sigmaE", "epsilon_sum", "sigmaG", "pi", "v", "betasqn")}
    s = [h.get_scalars(t) for t in range(c["traits"])]
    return {k: np.array([q[k] for q in s]) for k in ("epsilon_sum", "v", "betasqn")}


def run(state):
    c = state["case"]
    out = _run(state, c)
    if c["precision"] == "fp32":
        # the FP32 residual modes: a program that picks them keeps its samples in single precision
        out = _single(out)
    return out


def _single(v):
    if isinstance(v, dict):
        return {k: _single(x) for k, x in v.items()}
    if isinstance(v, list):
        return [_single(x) for x in v]
    return v.astype(np.float32) if isinstance(v, np.ndarray) and v.dtype == np.float64 else v


def _run(state, c):
    if c["kind"] == "decode":
        h = state["h"]
        h.load_bed(state["image"], LAYOUTS[c["layout"]])
        return h.marker_tables()
    if c["kind"] == "cohorts":
        hists, _ = brr.run_cohorts(state["hs"], state["seed"], state["it"], state["orders"])
        state["it"] += c["iterations"]
        return dict(hist=hists, state=[h.get_state() for h in state["hs"]])
    h = state["h"]
    if c["host"]:
        x = state["x"]
        _set_state(h, c, x)
        h.sweep(x["orders"][0], x["u"], x["z"])
        out = h.get_state()
        s = _scalars(h, c)
        return dict(out, epsilon_sum=s["epsilon_sum"], v=s["v"], betasqn=s["betasqn"])
    if c["start"] == "init":
        # a new analysis, from its first iteration
        _set_state(h, c, state["x"])
        hist = h.run_chain(state["seed"], 0, 0, state["x"]["orders"])
        return dict(h.get_state(), hist=hist)
    orders = state["orders"] if c["kind"] == "bayesw" else state["x"]["orders"]
    hist = h.run_chain(state["seed"], 0, state["it"], orders)
    state["it"] += c["iterations"]
    return dict(h.get_state(), hist=hist)


def work(case):
    c = case
    n, m, T, it = c["n"], c["m"], max(1, c["traits"]), c["iterations"]
    if c["kind"] == "decode":
        return {"bytes": 2 * m * ((n + 3) // 4) + 32 * m, "flops": 0}
    if c["kind"] == "cohorts":
        every = [work(d) for d in _cohorts(c)]
        return {k: sum(w[k] for w in every) for k in ("bytes", "flops")}
    cols = m * ((n + 3) // 4)
    if c["layout"] == "lists":
        cols = int(4 * n * m * (c["maf_lo"] + c["maf_hi"]))
    # the columns once per iteration, the residual in and out, the per-marker state in and out;
    # one multiply-add per individual, marker and trait
    return {"bytes": it * cols + 16 * n * T + 40 * m * T, "flops": 2.0 * n * m * T * it}


# ------------------------------------------------------------------- exact --

def _weights(c, codes):
    """Per marker and 2-bit value the dot's weight and the residual's change per unit of beta, and the sparse layouts'
    (mean, sd, Zsum, sqrdZ)."""
    n = float(c["n"])
    cnt = [(codes == v).sum(dim=1).double() for v in range(4)]
    two, miss, one = cnt[0], cnt[1], cnt[2]
    zero = torch.zeros_like(one)
    if c["layout"] == "dense":
        mean = (one + 2 * two) / (n - miss)
        cm = (one + 2 * two + miss * mean) / n
        d = torch.stack([2 - cm, mean - cm, 1 - cm, -cm], dim=1)
        ss = sum(cnt[v] * d[:, v] ** 2 for v in range(4))
        w = d / torch.sqrt(ss / (n - 1))[:, None]
        return w, w, None
    z, q = one + 2 * two, one + 4 * two
    mean = z / n
    if c["layout"] == "eigen":
        q, z = q + mean * mean * miss, z + mean * miss
    sd = torch.sqrt((q - 2 * mean * z + n * mean * mean) / (n - 1))
    w = torch.stack([zero + 2, mean if c["layout"] == "eigen" else zero, zero + 1, zero], dim=1)
    u = torch.stack([(2 - mean) / sd, zero, (1 - mean) / sd, -mean / sd], dim=1)
    return w, u, (mean, sd, z, q)


def exact(case, seed):
    """One exec in plain torch, 64 bits, one marker (or window) after the other; the chains draw their numbers
    from the package's own stream and have no value here."""
    c = dict(case)
    if c["kind"] == "decode":
        codes = _codes(c["n"], c["m"], c["maf_lo"], c["maf_hi"], c["miss"], seed)
        w, _, st = _weights(c, codes)
        if st is None:
            return w[:, [3, 2, 0, 1]]
        return torch.stack([st[0], st[1], st[3], st[2]], dim=1)
    if not c["host"]:
        return None
    dev = _dev()
    x = _bayesr_inputs(c, seed)
    codes = _codes(c["n"], c["m"], c["maf_lo"], c["maf_hi"], c["miss"], seed)
    w, u, st = _weights(c, codes)
    n, K, T = float(c["n"]), c["K"], max(1, c["traits"])

    def t64(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev, torch.float64)

    eps, beta = t64(x["eps"]).reshape(-1, T).clone(), t64(x["beta"]).reshape(-1, T).clone()
    uu, zz = t64(x["u"]).reshape(-1, T), t64(x["z"]).reshape(-1, T)
    comp = torch.from_numpy(x["comp"].astype(np.int64)).to(dev).reshape(-1, T).clone()
    acum_out = torch.zeros_like(beta)
    esum = eps.sum(dim=0)
    sE = x["sigmaE"]
    S, sG, pi = x["S"], x["sigmaG"], x["pi"]
    den = np.array([[n - 1 + sE / sG[g] / S[g][k] for k in range(K - 1)] for g in range(c["groups"])])
    c0 = np.array([[math.log(pi[g][0])] + [math.log(pi[g][k + 1]) - 0.5 * math.log(sG[g] / sE * (n - 1) * S[g][k] + 1)
                                           for k in range(K - 1)] for g in range(c["groups"])])
    den_t, c0_t = t64(den), t64(c0)
    half = torch.cat([torch.zeros(c["groups"], 1, dtype=torch.float64, device=dev), 0.5 / (den_t * sE)], dim=1)
    rden = torch.cat([torch.zeros(c["groups"], 1, dtype=torch.float64, device=dev), 1.0 / den_t], dim=1)
    bsd = torch.cat([torch.zeros(c["groups"], 1, dtype=torch.float64, device=dev), torch.sqrt(sE / den_t)], dim=1)
    v = torch.zeros((c["groups"], K, T), dtype=torch.float64, device=dev)
    bsq = torch.zeros((c["groups"], T), dtype=torch.float64, device=dev)
    ones = torch.ones((1, T), dtype=torch.float64, device=dev)
    group = x["group"]
    order = x["orders"][0].tolist()
    window = c["window"] or 1
    for a in range(0, c["m"], window):
        pend = []
        for j in order[a:a + window]:
            g = int(group[j])
            code = codes[j].int()
            dot = w[j].index_select(0, code) @ eps
            bo = beta[j].clone()
            if st is None:
                num = dot + bo * (n - 1)
            else:
                num = bo * (n - 1) - st[0][j] * esum / st[1][j] + dot / st[1][j]
            logl = c0_t[g][:, None] + half[g][:, None] * (num * num)[None, :]          # (K, T)
            diff = logl[None, :, :] - logl[:, None, :]                                 # [ref, i]
            p = 1.0 / torch.exp(diff).sum(dim=1)
            p = torch.where((diff[:, 1:].abs() > 700).any(dim=1), torch.zeros_like(p), p)
            cum = torch.cumsum(p, dim=0)
            sel = (uu[j][None, :] > cum).sum(dim=0)                                    # K: none
            none = sel >= K
            s1 = torch.where(none, torch.zeros_like(sel), sel)
            bn = torch.where(s1 > 0, zz[j] * bsd[g][s1] + num * rden[g][s1], torch.zeros_like(num))
            bn = torch.where(none, bo, bn)
            acum_out[j] = cum[0]
            beta[j] = bn
            comp[j] = torch.where(none, comp[j], sel)
            v[g].scatter_add_(0, s1[None, :], torch.where(none[None, :], 0 * ones, ones))
            bsq[g] += torch.where(s1 > 0, bn * bn, torch.zeros_like(bn))
            pend.append((j, code, bo - bn))
        for j, code, db in pend:
            eps += u[j].index_select(0, code)[:, None] * db[None, :]
            if st is not None:
                esum = esum + db * (st[2][j] - st[0][j] * n) / st[1][j]
    if st is None:
        esum = None                        # the dense model does not carry it
    vo = v.permute(2, 0, 1)
    out = dict(eps=eps, beta=beta, comp=comp.to(torch.int32), acum=acum_out)
    if c["traits"]:
        return dict(out, epsilon_sum=esum, v=vo, betasqn=bsq.t())
    return dict({k: q[:, 0] for k, q in out.items()}, epsilon_sum=None if esum is None else float(esum[0]), v=vo[0],
                betasqn=bsq[:, 0])
