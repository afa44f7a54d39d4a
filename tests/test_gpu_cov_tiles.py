"""The full-covariance likelihood at the edges of its matrix tiles: epoch counts
around multiples of 4 and 16 up to the largest, row counts around 16 (a wave)
and 64 (a workgroup), against the dense closed form (determinant lemma and
Woodbury's identity, no eigenbasis).  Tolerance 1e-10 relative, that of the
covariance tests at 16 epochs: the conditioning of the phase, not of the
rotation, sets it."""
import numpy as np
import pytest

from oracle import oracle
from thejoker_amd import device as D

pytestmark = pytest.mark.gpu


def _dense(t, rv, cov, trend, lam, t_ref, row, jitter):
    m = oracle.rv_unit(t, row[0], row[1], row[2], row[3], t_ref)
    X = np.column_stack([m, trend])
    Cs = cov + (row[4] ** 2 if jitter else 0.0) * np.eye(t.size)
    Ci = np.linalg.inv(Cs)
    G = np.diag(1 / lam) + X.T @ Ci @ X
    u = X.T @ Ci @ rv
    return -0.5 * (rv @ Ci @ rv - u @ np.linalg.solve(G, u) + t.size * np.log(2 * np.pi)
                   + np.linalg.slogdet(Cs)[1] + np.sum(np.log(lam)) + np.linalg.slogdet(G)[1])


@pytest.mark.parametrize("mode", ["physical", "reference"])
@pytest.mark.parametrize("N,L", [(1, 1), (3, 2), (4, 1), (5, 2), (15, 3), (16, 5), (17, 2), (31, 8),
                                 (32, 2), (33, 3), (48, 4), (49, 2), (63, 2), (64, 8)])
def test_cov_tiles(gpu, N, L, mode):
    g = np.random.default_rng(100 * N + L)
    t = np.sort(g.uniform(0, 400.0, N))
    err = g.uniform(0.1, 0.5, N)
    i = np.arange(N)
    cov = err[:, None] * 0.5 ** np.abs(i[:, None] - i[None, :]) * err[None, :]
    trend = np.column_stack([np.ones(N)] + [g.normal(size=N) for _ in range(L)])[:, :L - 1]
    lam = np.array([900.0] + [100.0] * (L - 1))
    rv = g.normal(0, 5, N)
    star = D.DeviceStar(t, rv, None, trend, np.zeros(L), lam, t[0], jitter_mode=mode, cov=cov)
    n = 1000
    rows = np.column_stack([np.exp(g.uniform(np.log(2), np.log(2048), n)), g.beta(0.867, 3.03, n),
                            g.uniform(0, 6.28, n), g.uniform(0, 6.28, n), np.exp(g.normal(-3, 1, n))])
    rows[17, 1] = 1 - 1e-9              # the fallback
    rows[20, 1] = 1.0                   # invalid
    full = D.lnl(star, D.PriorCache.from_packed(rows)).cpu().numpy()
    for k in [0, 1, 15, 16, 17, 63, 64, 65, 500, n - 1]:
        want = _dense(t, rv, cov, trend, lam, t[0], rows[k], mode == "physical")
        if k == 17:
            assert np.isfinite(full[k])          # ill-conditioned in the phase: finite is all
            continue
        assert abs(full[k] - want) <= 1e-10 * max(1.0, abs(want)), k
    assert np.isnan(full[20]) and np.isfinite(np.delete(full, 20)).all()
    # a row's value does not depend on its place or on its neighbours
    for m in (1, 15, 16, 17, 63, 64, 65, 999):
        part = D.lnl(star, D.PriorCache.from_packed(rows[:m])).cpu().numpy()
        assert np.array_equal(part, full[:m], equal_nan=True), m
    back = D.lnl(star, D.PriorCache.from_packed(rows[::-1].copy())).cpu().numpy()
    assert np.array_equal(back[::-1], full, equal_nan=True)
