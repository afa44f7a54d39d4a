"""Full-covariance stars of few epochs: a launch of many rows takes one lane
per row, one of few rows 16 rows a wave on the matrix cores.  Epoch counts
around 8, 16 and 24, at which the forms change, numbers of rows around the
lines: a row's lnL is the same bits in either, also where it needs the
bracketed Newton iteration or is invalid."""
import numpy as np
import pytest
import torch

from thejoker_amd import device as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["physical", "reference"])
@pytest.mark.parametrize("N,L", [(1, 1), (2, 8), (7, 2), (8, 6), (9, 4), (15, 3), (16, 5), (17, 6),
                                 (24, 7), (24, 8), (25, 6)])
def test_rows_same_bits(gpu, N, L, mode):
    g = np.random.default_rng(100 * N + L)
    t = np.sort(g.uniform(0, 400.0, N))
    err = g.uniform(0.1, 0.5, N)
    i = np.arange(N)
    cov = err[:, None] * 0.5 ** np.abs(i[:, None] - i[None, :]) * err[None, :]
    trend = np.column_stack([np.ones(N)] + [g.normal(size=N) for _ in range(L)])[:, :L - 1]
    lam = np.array([900.0] + [100.0] * (L - 1))
    star = D.DeviceStar(t, g.normal(0, 5, N), None, trend, np.zeros(L), lam, t[0],
                        jitter_mode=mode, cov=cov)
    n = 65537
    rows = np.column_stack([np.exp(g.uniform(np.log(2), np.log(2048), n)), g.beta(0.867, 3.03, n),
                            g.uniform(0, 6.28, n), g.uniform(0, 6.28, n), np.exp(g.normal(-3, 1, n))])
    rows[::97, 1] = 1 - 1e-9            # the fallback
    rows[5::101, 1] = 1.0               # invalid
    want = np.concatenate([D.lnl(star, D.PriorCache.from_packed(rows[k:k + 8192])).cpu().numpy()
                           for k in range(0, n, 8192)])
    assert np.isnan(want[5::101]).all() and np.isfinite(want).mean() > 0.98
    for m in (16384, 16385, 32769, 36865, 49153, 53249, 65536, n):
        full = D.lnl(star, D.PriorCache.from_packed(rows[:m])).cpu().numpy()
        assert np.array_equal(full, want[:m], equal_nan=True), m
    # over a row list, backwards
    idx = torch.arange(n - 1, -1, -1, device="cuda")
    back = D.lnl(star, D.PriorCache.from_packed(rows), rows=idx).cpu().numpy()
    assert np.array_equal(back, want[::-1], equal_nan=True)
