"""The linear posterior at the edges of its groups: epoch counts around the 16
lanes of a row, every number of linear parameters, row counts around a
workgroup (16 rows) and where a group takes several rows, against the normal
equations in NumPy (P >= 2 d, e < 0.95, 400 d: the phase is good to 1e-13 and
the design to 1e-11, so 1e-9 of the largest element holds with two digits to
spare), and the two launches against each other bit for bit."""
import numpy as np
import pytest

from oracle import oracle
from thejoker_amd import batch as B
from thejoker_amd import device as D

pytestmark = pytest.mark.gpu


def _cache(n, g):
    return [np.exp(g.uniform(np.log(2.0), np.log(500.0), n)), np.minimum(g.beta(0.867, 3.03, n), 0.95),
            g.uniform(0, 2 * np.pi, n), g.uniform(0, 2 * np.pi, n), g.uniform(0.0, 1.0, n)]


def _star(N, L, mode, g, cov=None):
    t = np.sort(g.uniform(0, 400.0, N))
    err = g.uniform(0.1, 0.5, N)
    trend = np.column_stack([np.ones(N)] + [g.normal(size=N) for _ in range(L)])[:, :L - 1]
    lam = np.array([900.0] + [100.0] * (L - 1))
    mu = np.linspace(0.5, -1.0, L)
    rv = g.normal(0, 5, N)
    C = np.diag(err ** 2)
    if cov:
        i = np.arange(N)
        C = err[:, None] * cov ** np.abs(i[:, None] - i[None, :]) * err[None, :]
    dev = D.DeviceStar(t, rv, None if cov else err ** -2.0, trend, mu, lam, t[0], jitter_mode=mode,
                       **(dict(cov=C) if cov else {}))
    return dev, (t, rv, C, trend, mu, lam)


def _check(case, cols, mode, rows, a, acov, ll):
    t, rv, C, trend, mu, lam = case
    for j, r in enumerate(rows):
        m = oracle.rv_unit(t, cols[0][r], cols[1][r], cols[2][r], cols[3][r], t[0], tol=1e-13)
        X = np.column_stack([m, trend])
        Cs = C + (cols[4][r] ** 2 if mode == "physical" else 0.0) * np.eye(t.size)
        Ci = np.linalg.inv(Cs)
        A = np.linalg.inv(np.diag(1 / lam) + X.T @ Ci @ X)
        a_ref = A @ (X.T @ Ci @ rv + mu / lam)
        d = rv - X @ mu
        Bc = Cs + (X * lam) @ X.T
        l_ref = -0.5 * (d @ np.linalg.solve(Bc, d) + t.size * np.log(2 * np.pi)
                        + np.linalg.slogdet(Bc)[1])
        assert np.abs(acov[j] - A).max() <= 1e-9 * np.abs(A).max()
        assert np.abs(a[j] - a_ref).max() <= 1e-9 * max(np.abs(a_ref).max(), 1.0)
        assert abs(ll[j] - l_ref) <= 1e-9 * max(abs(l_ref), 1.0)


@pytest.mark.parametrize("mode", ["physical", "reference"])
@pytest.mark.parametrize("N,L,cov", [(1, 1, 0), (15, 2, 0), (16, 3, 0), (17, 4, 0), (33, 5, 0),
                                     (64, 6, 0), (100, 7, 0), (200, 8, 0), (4, 2, 0.4),
                                     (17, 1, 0.4), (33, 3, 0.4), (64, 8, 0.4)])
def test_posterior_edges(gpu, N, L, cov, mode):
    g = np.random.default_rng(10 * N + L)
    cols = _cache(100, g)
    cache = D.PriorCache(*cols)
    star, case = _star(N, L, mode, g, cov)
    for k in (1, 15, 17):
        rows = g.choice(100, k, replace=False)
        _check(case, cols, mode, rows, *D.linear_posterior(star, cache, rows))


@pytest.mark.parametrize("k", [16383, 32768 + 5, 65536 + 17])
def test_posterior_many_rows(gpu, k):
    """Several rows per group: each row as in a launch of a few rows, and the
    star-table launch the same; an invalid row stays NaN by itself."""
    g = np.random.default_rng(k)
    cols = _cache(1000, g)
    cols[0][7] = np.nan
    cache = D.PriorCache(*cols)
    star, case = _star(20, 2, "physical", g)
    other, _ = _star(90, 2, "physical", g)
    rows = g.integers(0, 1000, k)
    rows[-1] = 7
    a, acov, ll = D.linear_posterior(star, cache, rows)
    a1, acov1, ll1 = D.linear_posterior(star, cache, np.arange(1000))
    assert np.array_equal(a, a1[rows], equal_nan=True)
    assert np.array_equal(acov, acov1[rows], equal_nan=True)
    assert np.array_equal(ll, ll1[rows], equal_nan=True)
    bad = rows == 7
    assert np.isnan(a[bad]).all() and np.isnan(ll[bad]).all() and np.isfinite(a[~bad]).all()
    pick = np.flatnonzero(~bad)[:5]
    _check(case, cols, "physical", rows[pick], a[pick], acov[pick], ll[pick])
    batch = B.StarBatch([star, other])
    got = D.posterior_inputs_table(batch, [1, 0], cache, [np.arange(500), rows])
    assert np.array_equal(got[1][1], a, equal_nan=True)
    assert np.array_equal(got[1][2], acov, equal_nan=True)
