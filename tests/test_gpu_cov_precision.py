"""Full-covariance likelihood, FP64: the weight 1 / (lambda + s^2) to an ulp.
One epoch with a residual so large, and priors so narrow, that the lnL is
-r^2 w / 2 to 1e-20: its relative error is the weight's plus the roundings of
s^2, lambda + s^2, w r, (w r) r and the final sums (each 2^-53, nine at most,
the weight's own at most two among them)."""
import numpy as np
import pytest

from thejoker_amd import device as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [1, 2])
def test_weight_to_an_ulp(gpu, L):
    g = np.random.default_rng(5)
    n = 4096
    s = np.exp(g.uniform(-3, 3, n))
    cache = D.PriorCache(np.full(n, 10.0), np.zeros(n), np.zeros(n), np.zeros(n), s)
    r, var = 1e9, 0.37
    star = D.DeviceStar(np.array([5e4]), np.array([r]), None, np.ones((1, L - 1)), np.zeros(L),
                        np.full(L, 1e-60), 5e4, jitter_mode="physical", cov=np.array([[var]]))
    v = np.longdouble(var) + s.astype(np.longdouble) ** 2
    want = -0.5 * (np.longdouble(r) ** 2 / v + np.log(2 * np.longdouble(np.pi)) + np.log(v))
    rel = np.abs((D.lnl(star, cache).cpu().numpy() - want) / want).astype(float)
    assert rel.max() <= 9 * 2.0 ** -53
