"""Few rows: the launches that spread a row's epochs over several lanes give
the bits of the launch with one row per lane (the many-star launch, which
evaluates every row that way), whatever the row count, the epoch count (whole
chunks, remainders, fewer epochs than lanes) and the number of linear
parameters; invalid rows stay NaN and rows that need the bracketed Newton
iteration take it.  The sums run in the same order with the same operations,
so the comparison is exact."""
import numpy as np
import pytest
import torch

from thejoker_amd import batch as B
from thejoker_amd import device as D

pytestmark = pytest.mark.gpu

TREND_VAR = [1e4, 0.25, 1e-6, 25.0, 25.0, 25.0, 25.0]


def _star(N, L, mode, seed=0):
    g = np.random.default_rng(seed + 1000 * N + L)
    t = np.sort(g.uniform(0, 900.0, N))
    dt = t - t[0]
    cols = [np.ones(N), dt, dt ** 2] + [(np.arange(N) % (j + 2) == 0) * 1.0 for j in range(4)]
    trend = np.stack(cols[:L - 1], axis=1) if L > 1 else np.zeros((N, 0))
    return D.DeviceStar(t, g.normal(0, 10, N), 1 / g.uniform(0.1, 0.5, N) ** 2, trend, np.zeros(L),
                        np.array([900.0] + TREND_VAR[:L - 1]), t[0], jitter_mode=mode)


def _cache(n, seed=1):
    g = np.random.default_rng(seed)
    P = np.exp(g.uniform(np.log(2), np.log(2048), n))
    e = g.beta(0.867, 3.03, n)
    s = np.exp(g.normal(-3, 1, n))
    P[3 % n::911] = 0.0                 # invalid
    e[5 % n::701] = 1.0 - 1e-9          # the fallback
    e[6 % n::1301] = 1.0                # invalid
    return D.PriorCache(P, e, g.uniform(0, 6.28, n), g.uniform(0, 6.28, n), s)


def _one_lane_per_row(star, cache, n, precision):
    table = B.StarBatch([star])
    items, _, total = B.work_items([n], 4096)
    bound = (torch.empty(n, dtype=torch.float32, device="cuda") if precision == "mixed" else None)
    ll = B.lnl_batch(table, cache, B.upload_items(items), len(items), total, precision, bound=bound)
    return ll.cpu().numpy(), None if bound is None else bound.cpu().numpy()


@pytest.mark.parametrize("mode", ["physical", "reference"])
@pytest.mark.parametrize("N,L", [(9, 2), (10, 2), (11, 1), (16, 3), (37, 5), (40, 2), (149, 3),
                                 (200, 8)])
def test_split_rows_are_the_same_bits(gpu, N, L, mode):
    star = _star(N, L, mode)
    big = 49153                          # one past the split's last row count
    cache = _cache(big)
    want, _ = _one_lane_per_row(star, cache, big, "f64")
    want_m, want_b = _one_lane_per_row(star, cache, big, "mixed")
    assert np.isnan(want).any() and np.isfinite(want).any()
    for n in (1, 7, 63, 64, 65, 1000, 4097, 20481, 33001, big - 1, big):
        got = D.lnl(star, cache, n=n).cpu().numpy()
        assert np.array_equal(got, want[:n], equal_nan=True), n
        b = torch.empty(n, dtype=torch.float32, device="cuda")
        got = D.lnl(star, cache, n=n, precision="mixed", bound=b).cpu().numpy()
        assert np.array_equal(got, want_m[:n], equal_nan=True), n
        assert np.array_equal(b.cpu().numpy(), want_b[:n]), n
    # a list of rows, and the maximum the rejection step takes from the launch
    rows = torch.as_tensor(np.random.default_rng(2).permutation(big)[:3001], device="cuda")
    got = D.lnl(star, cache, rows=rows).cpu().numpy()
    assert np.array_equal(got, want[rows.cpu().numpy()], equal_nan=True)
    state = D.pcg64_state(np.random.default_rng(3))
    fine = np.flatnonzero(np.isfinite(want))[:2999]
    _, idx, n_pass, mx = D.lnl_reject(star, cache, state, 64,
                                      rows=torch.as_tensor(fine, device="cuda"))
    assert mx == want[fine].max() and n_pass >= 1


@pytest.mark.parametrize("N,L", [(12, 2), (100, 3), (21, 5)])
@pytest.mark.parametrize("share", [0.001, 0.4, 1.0])
def test_scattered_rows_are_the_same_bits(gpu, N, L, share):
    """The FP64 re-evaluation of flagged rows of several segments, few (split
    over lanes) or many, writes the one-lane-per-row values and bound 0."""
    stars = [_star(N, L, "physical", seed=k) for k in range(3)]
    n = 30011
    cache = _cache(n, seed=5)
    table = B.StarBatch(stars)
    items, off, total = B.work_items([n] * 3, 4096)
    d_items = B.upload_items(items)
    want = B.lnl_batch(table, cache, d_items, len(items), total, "f64").cpu().numpy()
    ll = torch.full((total,), -1e9, dtype=torch.float64, device="cuda")
    g = np.random.default_rng(7)
    flagged = g.random(total) < share
    bound = torch.as_tensor(np.where(flagged, 1.0, 0.0).astype(np.float32), device="cuda")
    cnt = B.settle_tol_batch(table, cache, ll, bound, off, [n] * 3, tol=1e-3)
    got = ll.cpu().numpy()
    assert np.array_equal(got[flagged], want[flagged], equal_nan=True)
    assert (got[~flagged] == -1e9).all() and (bound.cpu().numpy() == 0).all()
    assert int(cnt.sum()) == flagged.sum()
