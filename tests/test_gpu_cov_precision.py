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


@pytest.mark.parametrize("scale", [1e-60, 1e60])
@pytest.mark.parametrize("N", [3, 17, 40])
def test_variances_far_from_one(gpu, N, scale):
    """The product of the variances passes the exponent range within a few
    epochs; the sum of their logarithms does not.  Data, priors and jitter in
    units of `scale` shift the lnL by -N ln(scale), up to the rounding of the
    sum of the logarithms.  (Past 1e77 the squares in the system's own determinant
    leave the range.)"""
    g = np.random.default_rng(N)
    n = 256
    t = np.sort(g.uniform(0, 300.0, N))
    err = g.uniform(0.1, 0.5, N)
    C = err[:, None] * 0.6 ** np.abs(np.arange(N)[:, None] - np.arange(N)) * err[None, :]
    rv, s = g.normal(0, 3, N), np.exp(g.normal(-3, 1, n))
    cols = [np.exp(g.uniform(1, 6, n)), g.beta(0.867, 3.03, n), g.uniform(0, 6.28, n),
            g.uniform(0, 6.28, n)]
    ll = []
    for q in (1.0, scale):
        star = D.DeviceStar(t, rv * q, None, np.ones((N, 1)), np.zeros(2),
                            np.array([900.0, 1e4]) * q * q, t[0], jitter_mode="physical",
                            cov=C * q * q)
        ll.append(D.lnl(star, D.PriorCache(*cols, s * q)).cpu().numpy())
    shift = N * np.log(scale)
    assert np.isfinite(ll[0]).all()
    np.testing.assert_allclose(ll[1], ll[0] - shift, rtol=0, atol=1e-12 * abs(shift))
