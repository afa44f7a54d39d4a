"""Timing cases: the calls a user of this package has it do, over the sizes,
options and precisions they are used at.

Each case is a dict of plain values with a ``kind``:

* ``lnl``        marginal lnL of prior rows of one star (``device.lnl``): the
                 first rounds of an iterative run, chunks, whole caches; FP64
                 or mixed; sampled jitter or none; trends, survey offsets,
                 a FixedCompanionMass K prior.
* ``lnl_cov``    the same for data with a full covariance.
* ``reject``     lnL and rejection step of one star in one call
                 (``device.lnl_reject``), the FP64 ``rejection_sample``.
* ``settle``     the mixed-precision ``rejection_sample``: mixed lnL with its
                 bounds, FP64 settling, rejection step.
* ``prune``      the probe-bounded ``rejection_sample`` of a star with many
                 epochs (``batch.prune_reject_batch``).
* ``many``       many stars against one shared cache: one persistent launch,
                 then every star's rejection step.
* ``posterior``  linear parameters of accepted rows
                 (``device.linear_posterior``).
* ``iterative``  a whole ``TheJoker.iterative_rejection_sample`` call, from
                 RVData to JokerSamples.

Sizes: 16 epochs and 2^24 rows, 50 epochs, 3 to 64 epochs for many stars, up
to 200 epochs, 128 x the requested samples for a first round and 256 kept
samples are those of bench.py and the package's own defaults; the prior is
the default one (P log-uniform, e ~ Beta(0.867, 3.03), uniform angles, ln s
normal when the jitter is sampled).
"""
import math

import numpy as np
import torch

from thejoker_amd import _lib
from thejoker_amd import batch as B
from thejoker_amd import device as D
from thejoker_amd import units as u
from thejoker_amd.data import RVData
from thejoker_amd.distributions import Normal
from thejoker_amd.prior import JokerPrior
from thejoker_amd.thejoker import TheJoker

T0 = 58000.0          # BMJD of the first possible epoch
V0_VAR, K_VAR = 1e4, 900.0
OFFSET_VAR = 25.0
# variance of the k-th trend coefficient (km/s / day^k), k = 1, 2, ...
TREND_VAR = {1: 0.25, 2: 1e-6, 3: 1e-12}
FCM = dict(k_prior_mode=_lib.JK_KPRIOR_FIXED_COMPANION_MASS, sigma_K0=30.0, P0=365.25, max_K=500.0)
# rows x epochs of the largest listed case, and of the largest drawn one
MAX_WORK = 64 * (1 << 18) * 34


def listed():
    return [
        # The first round of an iterative run that wants 16 samples (128 x 16
        # rows) on a typical star: the smallest likelihood call, all latency.
        dict(name="lnl_first_round", kind="lnl", n=2048, m=16, poly=1, offsets=0, jitter=True,
             fcm=False, precision="f64"),
        # The first round for 256 samples (128 x 256 rows, and a ragged rest)
        # on a well observed star with a linear trend.
        dict(name="lnl_round_long_star", kind="lnl", n=33001, m=149, poly=2, offsets=0, jitter=True,
             fcm=False, precision="f64"),
        # A chunk of a prior cache for a star of three surveys with a linear
        # trend, the default prior's K and no jitter: five linear parameters.
        dict(name="lnl_three_surveys", kind="lnl", n=1 << 20, m=37, poly=2, offsets=2, jitter=False,
             fcm=True, precision="f64"),
        # The mixed-precision likelihood of a 50-epoch star with its bounds.
        dict(name="lnl_mixed_m50", kind="lnl", n=1 << 22, m=50, poly=1, offsets=0, jitter=True,
             fcm=False, precision="mixed"),
        # Correlated noise: RVs with a full covariance matrix.
        dict(name="lnl_full_covariance", kind="lnl_cov", n=1 << 18, m=40, poly=1, offsets=0,
             jitter=True, fcm=False, precision="f64"),
        # rejection_sample at the benchmark's size: 16 epochs, 2^24 rows.
        dict(name="reject_2p24", kind="reject", n=1 << 24, m=16, poly=1, offsets=0, jitter=True,
             fcm=False, precision="f64", keep=256, binary=True),
        # The same call in mixed precision on a quarter of the rows.
        dict(name="settle_2p22", kind="settle", n=1 << 22, m=16, poly=1, offsets=0, jitter=True,
             fcm=False, precision="mixed", keep=256, binary=True),
        # rejection_sample with probe bounds on a star of 100 epochs.
        dict(name="prune_m100", kind="prune", n=1 << 21, m=100, poly=1, offsets=0, jitter=True,
             fcm=False, precision="f64", keep=256, binary=True),
        # A survey's stars in mixed precision, half of them constant (flat
        # likelihoods, every row in reach of the maximum).
        dict(name="many_mixed", kind="many", n=1 << 18, stars=64, m_lo=3, m_hi=64, poly=2,
             offsets=0, jitter=True, fcm=False, precision="mixed", keep=256),
        # Few rows for each of many sparsely observed stars, in FP64.
        dict(name="many_f64_sparse", kind="many", n=50000, stars=96, m_lo=3, m_hi=12, poly=1,
             offsets=0, jitter=False, fcm=False, precision="f64", keep=256),
        # Linear parameters of 2048 accepted rows (eight stars' worth).
        dict(name="posterior_2048", kind="posterior", n=1 << 18, k=2048, m=64, poly=2, offsets=0,
             jitter=True, fcm=False, precision="f64"),
        # A whole iterative run, RVData to samples.
        dict(name="iterative_64", kind="iterative", n=1 << 20, m=6, poly=1, offsets=0,
             jitter=False, fcm=False, precision="f64", requested=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["lnl", "lnl", "lnl", "lnl_cov", "reject", "settle", "prune", "many",
                       "posterior", "iterative"])
    c = dict(kind=kind, poly=rng.choice([1, 1, 2, 3]), offsets=rng.choice([0, 0, 1, 2]),
             jitter=rng.random() < 0.6, fcm=rng.random() < 0.3, precision="f64")
    m = _log_int(rng, 3, 200)
    if kind == "lnl":
        c.update(precision=rng.choice(["f64", "f64", "mixed"]), m=m,
                 n=_log_int(rng, 1000, min(1 << 23, MAX_WORK // m)))
    elif kind == "lnl_cov":
        m = rng.randint(4, 64)
        c.update(m=m, n=_log_int(rng, 1000, 1 << 19))
    elif kind in ("reject", "settle"):
        m = _log_int(rng, 4, 100)
        c.update(m=m, n=_log_int(rng, 4000, min(1 << 24, MAX_WORK // m)), keep=256,
                 binary=rng.random() < 0.6, precision="f64" if kind == "reject" else "mixed")
    elif kind == "prune":
        m = _log_int(rng, 20, 200)
        c.update(m=m, n=_log_int(rng, 100000, min(1 << 22, MAX_WORK // m)), keep=256, binary=True,
                 precision=rng.choice(["f64", "mixed"]))
    elif kind == "many":
        stars = rng.randint(16, 128)
        lo, hi = rng.choice([(3, 64), (3, 12), (8, 33)])
        c.update(stars=stars, m_lo=lo, m_hi=hi, keep=256, precision=rng.choice(["f64", "mixed"]),
                 n=_log_int(rng, 2000, min(1 << 18, MAX_WORK // (stars * (lo + hi) // 2))))
    elif kind == "posterior":
        c.update(m=m, k=_log_int(rng, 16, 4096), n=1 << 16)
    else:
        # the sampler's own API with the constant-velocity trend
        c.update(m=rng.randint(4, 8), n=_log_int(rng, 200000, 1 << 20), requested=rng.choice([16, 64, 256]),
                 poly=1, offsets=0, jitter=False, fcm=False)
    return c


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------
def _n_linear(c):
    return 1 + c["poly"] + c["offsets"]


def _kepler_np(x, e):
    E = x + e * np.sin(x)
    for _ in range(60):
        E = E - (E - e * np.sin(E) - x) / (1 - e * np.cos(E))
    return E


def _star(c, m, rng, binary=True):
    """Plain arrays of one star of m epochs: times, RVs, errors, the trend
    columns [1, survey indicators, dt, dt^2, ...], prior means and variances."""
    span = rng.uniform(200.0, 3000.0)
    t = T0 + np.sort(rng.uniform(0.0, span, m))
    err = rng.uniform(0.1, 0.5, m)
    t_ref = t.min()
    dt = t - t_ref
    v0 = rng.normal(0.0, 30.0)
    rv = np.full(m, v0)
    P = math.exp(rng.uniform(math.log(2.0), math.log(2048.0)))
    e, om, M0 = rng.beta(0.867, 3.03), rng.uniform(0, 2 * np.pi), rng.uniform(0, 2 * np.pi)
    K = rng.uniform(3.0, 30.0) * (1.0 if binary else 0.0)
    x = np.mod(2 * np.pi * dt / P - M0 + np.pi, 2 * np.pi) - np.pi
    E = _kepler_np(x, e)
    f = 2 * np.arctan2(np.sqrt(1 + e) * np.sin(E / 2), np.sqrt(1 - e) * np.cos(E / 2))
    rv = rv + K * (np.cos(om + f) + e * np.cos(om))
    survey = np.arange(m) % (c["offsets"] + 1)
    cols = [np.ones(m)]
    lam = [K_VAR, V0_VAR]
    for i in range(c["offsets"]):
        ind = (survey == i + 1).astype(np.float64)
        cols.append(ind)
        lam.append(OFFSET_VAR)
        rv = rv + rng.normal(0.0, 2.0) * ind
    for k in range(1, c["poly"]):
        cols.append(dt ** k)
        lam.append(TREND_VAR[k])
        rv = rv + rng.normal(0.0, 0.1 * math.sqrt(TREND_VAR[k])) * dt ** k
    rv = rv + rng.normal(0.0, err)
    return dict(t=t, rv=rv, err=err, t_ref=t_ref, trend=np.stack(cols, axis=1),
                mu=np.zeros(len(lam)), lam=np.array(lam))


def _cov(err, rho=0.6):
    i = np.arange(err.size)
    return err[:, None] * rho ** np.abs(i[:, None] - i[None, :]) * err[None, :]


def _prior_columns(c, seed):
    """P, e, omega, M0, s as CPU float64 tensors, drawn on the GPU from seed."""
    n = c["n"]
    with torch.random.fork_rng(devices=[0]):
        torch.manual_seed(seed)
        dev = torch.device("cuda", 0)
        kw = dict(dtype=torch.float64, device=dev)
        P = torch.exp(torch.rand(n, **kw) * math.log(2048.0 / 2.0) + math.log(2.0))
        ab = torch.tensor([0.867, 3.03], **kw)
        e = torch.distributions.Beta(ab[0], ab[1]).sample((n,)).clamp_(max=0.999999)
        om = torch.rand(n, **kw) * (2 * math.pi)
        M0 = torch.rand(n, **kw) * (2 * math.pi)
        s = torch.exp(torch.randn(n, **kw) - 3.0) if c["jitter"] else torch.zeros(n, **kw)
        return [x.cpu() for x in (P, e, om, M0, s)]


def _inputs(c, seed):
    """(stars, prior columns, numpy generator for the rest) of a case."""
    rng = np.random.default_rng(seed)
    if c["kind"] == "many":
        ms = rng.integers(c["m_lo"], c["m_hi"] + 1, c["stars"])
        stars = [_star(c, int(m), rng, binary=i % 2 == 0) for i, m in enumerate(ms)]
    else:
        stars = [_star(c, c["m"], rng, binary=c.get("binary", True))]
    return stars, _prior_columns(c, seed), rng


def _device_star(c, st):
    kw = FCM if c["fcm"] else {}
    cov = _cov(st["err"]) if c["kind"] == "lnl_cov" else None
    ivar = None if cov is not None else 1.0 / st["err"] ** 2
    return D.DeviceStar(st["t"], st["rv"], ivar, st["trend"], st["mu"], st["lam"], st["t_ref"],
                        jitter_mode=_jitter_mode(c), cov=cov, **kw)


def _jitter_mode(c):
    return "physical" if c["jitter"] else "reference"


def _pcg(rng):
    return D.pcg64_state(np.random.default_rng(int(rng.integers(1 << 62))))


def prepare(case, seed):
    """What a user's program holds before the call: the prior cache on the
    device, the star (or star table and its work items), the random stream."""
    c = case
    stars, cols, rng = _inputs(c, seed)
    cache = D.PriorCache(*[x.numpy() for x in cols])
    state = dict(case=c, cache=cache)
    if c["kind"] == "iterative":
        st = stars[0]
        state.update(
            seed=seed,
            data=RVData(st["t"], u.Quantity(st["rv"], u.km / u.s), u.Quantity(st["err"], u.km / u.s)),
            prior=JokerPrior.default(P_min=2 * u.day, P_max=2048 * u.day, sigma_v=100 * u.km / u.s,
                                     pars={"K": Normal(0.0, 30.0, unit=u.km / u.s)}))
        return state
    dstars = [_device_star(c, st) for st in stars]
    state.update(stars=dstars, star=dstars[0])
    if c["kind"] in ("reject", "settle", "prune", "many"):
        state["streams"] = [_pcg(rng) for _ in dstars]
        state["sizes"] = np.full(len(dstars), c["n"])
    if c["kind"] in ("settle", "prune", "many"):
        state["table"] = B.StarBatch(dstars)
    if c["kind"] in ("prune", "many"):
        shape = state["shape"] = B.LaunchShape()
        items, off, total = B.work_items(state["sizes"], shape.tile)
        items = items[B.heaviest_first(items, state["table"].M)]
        state.update(items=B.upload_items(items), n_items=len(items), off=off, total=total)
    if c["kind"] == "prune":
        probe, add = D.probe_star(dstars[0].arrays(), jitter_mode=_jitter_mode(c))
        state.update(probes=B.StarBatch([probe]), adds=np.array([add]), probed=np.array([True]))
    if c["kind"] == "posterior":
        state["rows"] = np.sort(rng.choice(c["n"], size=min(c["k"], c["n"]), replace=False))
    return state


def _filled(a, n, value):
    """a with `value` appended up to n entries: how many rows are accepted
    depends on the inputs, the shape of the outputs does not."""
    out = np.full(n, value, dtype=a.dtype)
    out[:len(a)] = a
    return out


def run(state):
    """One pass; see the kinds in the module's docstring."""
    c, cache = state["case"], state["cache"]
    kind, n = c["kind"], c["n"]
    if kind in ("lnl", "lnl_cov"):
        if c["precision"] == "f64":
            return {"ll": D.lnl(state["star"], cache)}
        bound = torch.empty(n, dtype=torch.float32, device=cache.P.device)
        ll = D.lnl(state["star"], cache, precision="mixed", bound=bound)
        return {"ll": ll, "bound": bound}
    if kind == "reject":
        ll, idx, n_pass, mx = D.lnl_reject(state["star"], cache, state["streams"][0], c["keep"])
        return {"ll": ll, "idx": _filled(idx, c["keep"], -1), "n_pass": n_pass, "llmax": mx}
    if kind == "settle":
        bound = torch.empty(n, dtype=torch.float32, device=cache.P.device)
        ll = D.lnl(state["star"], cache, precision="mixed", bound=bound)
        idx, n_pass, mx, _ = B.settle_reject_batch(state["table"], cache, ll, bound, [0], [n],
                                                   state["streams"], c["keep"])
        return {"ll": ll, "idx": _filled(idx[0], c["keep"], -1), "n_pass": n_pass, "llmax": mx}
    if kind == "prune":
        ll, bound, res, _ = B.prune_reject_batch(state["table"], state["probes"], state["adds"],
                                                 state["probed"], cache, state["items"],
                                                 state["n_items"], state["off"], state["sizes"],
                                                 state["streams"], c["keep"], c["precision"],
                                                 state["shape"])
        return {"idx": _filled(res[0][0], c["keep"], -1), "n_pass": res[1], "llmax": res[2],
                "ll": ll, "bound": bound}
    if kind == "many":
        if c["precision"] == "f64":
            ll = B.lnl_batch(state["table"], cache, state["items"], state["n_items"],
                             state["total"], "f64", state["shape"])
            idx, n_pass, mx = B.reject_batch(ll, state["off"], state["sizes"], state["streams"],
                                             c["keep"])
        else:
            bound = torch.empty(state["total"], dtype=torch.float32, device=cache.P.device)
            ll = B.lnl_batch(state["table"], cache, state["items"], state["n_items"],
                             state["total"], "mixed", state["shape"], bound=bound)
            idx, n_pass, mx, _ = B.settle_reject_batch(state["table"], cache, ll, bound,
                                                       state["off"], state["sizes"],
                                                       state["streams"], c["keep"])
        return {"ll": ll, "idx": _filled(np.concatenate(idx), c["stars"] * c["keep"], -1),
                "n_pass": n_pass, "llmax": mx}
    if kind == "posterior":
        a, cov, ll = D.linear_posterior(state["star"], cache, state["rows"])
        return {"a": a, "cov": cov, "ll": ll}
    joker = TheJoker(state["prior"], rng=np.random.default_rng(state["seed"]),
                     precision=c["precision"])
    out = joker.iterative_rejection_sample(state["data"], cache, c["requested"], in_memory=True)
    return {k: _filled(v.value, c["requested"], 0.0) for k, v in out.tbl.items()}


# ---------------------------------------------------------------------------
# What a pass cannot do without.
# ---------------------------------------------------------------------------
def _f_epoch(c, L):
    """Operations per row and epoch: Kepler solve, design column and the
    moments of L linear parameters (add and multiply 1, fused 2, divide 4,
    sin / cos 8), with the jitter weights when the jitter is sampled."""
    return 156 + (20 if c["jitter"] else 0) + 8 * max(L - 2, 0)


def work(case):
    c = case
    L, n, kind = _n_linear(c), c["n"], c["kind"]
    cols = 40 if c["jitter"] else 32
    per_row = 90 + 38 * max(L - 2, 0)
    if kind == "many":
        m = (c["m_lo"] + c["m_hi"]) / 2
        rows = n * c["stars"]
        return {"bytes": float(cols * n + 8 * rows),
                "flops": float(rows) * (m * _f_epoch(c, L) + per_row)}
    if kind == "posterior":
        k = min(c["k"], n)
        return {"bytes": float(k * (40 + 8 + 8 * (L + L * L + 1))),
                "flops": float(k) * (c["m"] * _f_epoch(c, L) + per_row)}
    if kind == "prune":
        # the probe of about sqrt(m) epochs on every row
        m = max(5, min(16, round(math.sqrt(c["m"]))))
        return {"bytes": float(n * (cols + 12)), "flops": float(n) * (m * _f_epoch(c, L) + per_row)}
    if kind == "iterative":
        # the first round; how many follow depends on the star
        rows = min(n, 128 * c["requested"])
        return {"bytes": float(rows * (cols + 8)),
                "flops": float(rows) * (c["m"] * _f_epoch(c, L) + per_row)}
    fl = float(n) * (c["m"] * _f_epoch(c, L) + per_row)
    if kind == "lnl_cov":
        fl += 2.0 * n * c["m"] ** 2
    out = 8 + (4 if c["precision"] == "mixed" and kind == "lnl" else 0)
    return {"bytes": float(n * (cols + out)), "flops": fl}


# ---------------------------------------------------------------------------
# The same numbers in plain 64-bit torch.
# ---------------------------------------------------------------------------
def _design(dt, P, e, om, M0):
    """cos(omega + f) + e cos omega for rows x epochs.  The phase is reduced
    with fmod, which is exact; Newton from Danby's start converges for every
    e < 1."""
    x = torch.fmod(dt[None, :], P[:, None]) / P[:, None] * (2 * math.pi) - M0[:, None]
    k = torch.round(x / (2 * math.pi))
    x = (x - k * 6.283185307179586) - k * 2.4492935982947064e-16
    ax = x.abs()
    ee = e[:, None]
    E = torch.clamp(ax + 0.85 * ee, max=math.pi)
    for _ in range(40):
        d = (E - ee * torch.sin(E) - ax) / (1 - ee * torch.cos(E))
        E = E - d
        if float(d.abs().max()) < 1e-14:
            break
    sE, cE = torch.sin(E) * torch.sign(x), torch.cos(E)
    den = 1 - ee * cE
    cf, sf = (cE - ee) / den, torch.sqrt(1 - ee * ee) * sE / den
    return torch.cos(om)[:, None] * (cf + ee) - torch.sin(om)[:, None] * sf


def _exact_rows(c, st, cols, clip=True):
    """lnL, posterior mean and covariance of the linear parameters for the
    rows in cols (CUDA float64), in chunks."""
    dev = cols[0].device
    dt = torch.as_tensor(st["t"] - st["t_ref"], device=dev)
    y = torch.as_tensor(st["rv"], device=dev)
    T = torch.as_tensor(st["trend"], device=dev)
    lam_t = torch.as_tensor(st["lam"], device=dev)
    sig2 = torch.as_tensor(st["err"] ** 2, device=dev)
    Q = None
    if c["kind"] == "lnl_cov":
        ev, V = np.linalg.eigh(_cov(st["err"]))
        sig2, Q = torch.as_tensor(ev, device=dev), torch.as_tensor(V, device=dev)
        y, T = Q.T @ y, Q.T @ T
    N, L = T.shape[0], T.shape[1] + 1
    step = max(1, (1 << 24) // (N * max(L, 4)))
    lls, means, covs = [], [], []
    for lo in range(0, cols[0].shape[0], step):
        P, e, om, M0, s = [x[lo:lo + step] for x in cols]
        m = _design(dt, P, e, om, M0)
        if Q is not None:
            m = m @ Q.contiguous()
        v = sig2[None, :] + (s * s)[:, None] if c["jitter"] else sig2[None, :].expand(m.shape)
        X = torch.cat([m[:, :, None], T[None].expand(m.shape[0], N, L - 1)], dim=2)
        lam = lam_t[None, :].repeat(m.shape[0], 1)
        if c["fcm"]:
            l0 = FCM["sigma_K0"] ** 2 / ((1 - e * e) * (P / FCM["P0"]) ** (2.0 / 3.0))
            lam[:, 0] = torch.clamp(l0, max=FCM["max_K"] ** 2) if clip else l0
        # the least-squares form: rows weighted by 1 / sigma, the prior as L
        # further rows; its QR does not square the condition number
        sw = 1.0 / torch.sqrt(v)
        A = torch.cat([X * sw[:, :, None], torch.diag_embed(1.0 / torch.sqrt(lam))], dim=1)
        b = torch.cat([y[None, :] * sw, torch.zeros_like(lam)], dim=1)
        R = _qr_r(torch.cat([A, b[:, :, None]], dim=2))
        Rl, z = R[:, :L, :L], R[:, :L, L]
        chi2 = R[:, L, L] ** 2
        logdet = 2 * torch.log(torch.diagonal(Rl, dim1=1, dim2=2).abs()).sum(1)
        lls.append(-0.5 * (chi2 + N * math.log(2 * math.pi) + torch.log(v).sum(1)
                           + torch.log(lam).sum(1) + logdet))
        if c["kind"] == "posterior":
            Ri = torch.linalg.solve_triangular(Rl, torch.eye(L, dtype=Rl.dtype, device=dev)
                                               .expand(Rl.shape).contiguous(), upper=True)
            means.append((Ri * z[:, None, :]).sum(2))
            covs.append((Ri[:, :, None, :] * Ri[:, None, :, :]).sum(3))
    cat = lambda xs: torch.cat(xs) if xs else None
    return cat(lls), cat(means), cat(covs)


def _qr_r(A):
    """Upper triangular factor of each matrix of a stack (rows x m x k, k
    small), by modified Gram-Schmidt with a second pass."""
    A = A.clone()
    k = A.shape[2]
    R = torch.zeros(A.shape[0], k, k, dtype=A.dtype, device=A.device)
    for j in range(k):
        for _ in range(2):
            for i in range(j):
                r = (A[:, :, i] * A[:, :, j]).sum(1)
                R[:, i, j] += r
                A[:, :, j] -= r[:, None] * A[:, :, i]
        nrm = torch.sqrt((A[:, :, j] ** 2).sum(1))
        R[:, j, j] = nrm
        A[:, :, j] /= nrm[:, None]
    return R


def exact(case, seed):
    """What run() returns, from plain 64-bit torch; None for indices and
    counts, for error bounds and for random draws."""
    c = case
    if c["kind"] in ("iterative", "prune"):
        # draws of the linear parameters; a buffer that holds upper bounds
        # for most rows
        return None
    if c["kind"] == "many" and c["stars"] * c["n"] * c["m_hi"] > 1 << 29:
        return None
    stars, cols, rng = _inputs(c, seed)
    cols = [x.cuda() for x in cols]
    if c["kind"] == "posterior":
        rows = torch.as_tensor(np.sort(rng.choice(c["n"], size=min(c["k"], c["n"]), replace=False)),
                               device="cuda")
        ll, a, cov = _exact_rows(c, stars[0], [x[rows] for x in cols], clip=False)
        return {"a": a.cpu().numpy(), "cov": cov.cpu().numpy(), "ll": ll.cpu().numpy()}
    lls = [_exact_rows(c, st, cols)[0] for st in stars]
    if c["kind"] in ("lnl", "lnl_cov"):
        out = {"ll": lls[0]}
        if c["precision"] == "mixed":
            out["bound"] = None
        return out
    mx = [float(x.max()) for x in lls]
    if c["kind"] == "reject":
        return {"ll": lls[0], "idx": None, "n_pass": None, "llmax": mx[0]}
    return {"ll": torch.cat(lls), "idx": None, "n_pass": None, "llmax": np.array(mx)}
