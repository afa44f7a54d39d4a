"""Row counts on both sides of the lines between the FP64 likelihood's launches
(a row's epochs over several lanes; at most one wave per SIMD; more) and of the
mixed one's: the same bits as the many-star launch, for epoch counts with every
remainder of four, with and without jitter, with and without a first trend
column of ones; the rejection step's maximum with them."""
import numpy as np
import pytest
import torch

from thejoker_amd import batch as B
from thejoker_amd import device as D

pytestmark = pytest.mark.gpu

ROWS = 65537 + 63


def _split_line(N, mixed):
    if not mixed:
        return 0 if N < 10 else min(36864, 600 * (N - 3))
    if N < 30:
        return 0 if N < 17 else 2048
    return min(49152, max(20480, 490 * N))


@pytest.fixture(scope="module")
def cache(gpu):
    g = np.random.default_rng(11)
    P = np.exp(g.uniform(np.log(2), np.log(2048), ROWS))
    e = g.beta(0.867, 3.03, ROWS)
    P[3::911] = 0.0                     # invalid
    e[5::701] = 1.0 - 1e-9              # the fallback
    e[6::1301] = 1.0                    # invalid
    return D.PriorCache(P, e, g.uniform(0, 6.28, ROWS), g.uniform(0, 6.28, ROWS),
                        np.exp(g.normal(-3, 1, ROWS)))


def _star(N, L, mode, ones):
    g = np.random.default_rng(1000 * N + L)
    t = np.sort(g.uniform(0, 900.0, N))
    cols = [np.ones(N) if ones else 1.0 + 0.1 * np.cos(t), t - t[0], g.normal(0, 1, N),
            g.normal(0, 1, N), g.normal(0, 1, N), g.normal(0, 1, N), g.normal(0, 1, N)]
    trend = np.stack(cols[:L - 1], axis=1) if L > 1 else np.zeros((N, 0))
    return D.DeviceStar(t, g.normal(0, 10, N), 1 / g.uniform(0.1, 0.5, N) ** 2, trend, np.zeros(L),
                        np.array([900.0, 1e4, 0.25, 25.0, 25.0, 25.0, 25.0, 25.0])[:L], t[0],
                        jitter_mode=mode)


@pytest.mark.parametrize("mode", ["physical", "reference"])
@pytest.mark.parametrize("N,L,ones", [(1, 1, True), (3, 2, True), (4, 3, False), (9, 3, True),
                                      (10, 2, True), (16, 2, False), (17, 4, True), (18, 3, True),
                                      (29, 2, True), (30, 5, True), (47, 6, True), (64, 3, True),
                                      (101, 8, True), (110, 2, True)])
def test_same_bits_on_both_sides(cache, N, L, ones, mode):
    star = _star(N, L, mode, ones)
    table = B.StarBatch([star])
    items, _, total = B.work_items([ROWS], 4096)
    d_items = B.upload_items(items)
    want = B.lnl_batch(table, cache, d_items, len(items), total, "f64").cpu().numpy()
    bound = torch.empty(ROWS, dtype=torch.float32, device="cuda")
    want_m = B.lnl_batch(table, cache, d_items, len(items), total, "mixed",
                         bound=bound).cpu().numpy()
    want_b = bound.cpu().numpy()
    ok = np.isfinite(want)
    assert ok.any() and np.isnan(want).any()
    for n in {max(_split_line(N, False), 1), _split_line(N, False) + 1, 49153, 65535, 65536, 65537,
              ROWS}:
        got = D.lnl(star, cache, n=n).cpu().numpy()
        assert np.array_equal(got, want[:n], equal_nan=True), n
    for n in {max(_split_line(N, True), 1), _split_line(N, True) + 1, 65536}:
        b = torch.empty(n, dtype=torch.float32, device="cuda")
        got = D.lnl(star, cache, n=n, precision="mixed", bound=b).cpu().numpy()
        assert np.array_equal(got, want_m[:n], equal_nan=True), n
        assert np.array_equal(b.cpu().numpy(), want_b[:n]), n
    fine = np.flatnonzero(ok)[:60001]
    state = D.pcg64_state(np.random.default_rng(3))
    _, _, n_pass, mx = D.lnl_reject(star, cache, state, 64,
                                    rows=torch.as_tensor(fine, device="cuda"))
    assert mx == want[fine].max() and n_pass >= 1


@pytest.mark.parametrize("N,L", [(3, 2), (8, 2), (9, 3), (12, 2), (30, 5), (55, 4), (56, 5),
                                 (87, 2), (88, 3)])
@pytest.mark.parametrize("slots", [False, True])
def test_scatter_line(cache, N, L, slots):
    """FP64 re-evaluations on both sides of the line where a row's epochs are
    spread over lanes (4 (N - 8) waves of 64, 320 or 192 at most): the rows' own values,
    bounds 0 and counts, for tables of stars and of slots."""
    star = _star(N, L, "physical", True)
    table = B.StarBatch([star])
    items, off, total = B.work_items([ROWS], 4096)
    d_items = B.upload_items(items)
    want = B.lnl_batch(table, cache, d_items, len(items), total, "f64").cpu().numpy()
    if slots:
        table = B.StarBatch.slots(2, L, "physical")
        table.set(1, star)
    waves = min(max(4 * (N - 8), 0), 320 if L <= 3 else 192)
    g = np.random.default_rng(N)
    for n in sorted({1, max(64 * waves, 1), 64 * waves + 1}):
        at = np.sort(g.permutation(ROWS)[:n])
        b = np.zeros(ROWS, dtype=np.float32)
        b[at] = 1.0
        ll = torch.full((ROWS,), -1e9, dtype=torch.float64, device="cuda")
        bound = torch.as_tensor(b, device="cuda")
        cnt = B.settle_tol_batch(table, cache, ll, bound, [0], [ROWS], stars=[int(slots)], tol=1e-3)
        got = ll.cpu().numpy()
        assert int(cnt[0]) == n and (bound.cpu().numpy() == 0).all()
        assert np.array_equal(got[at], want[at], equal_nan=True)
        assert (np.delete(got, at) == -1e9).all()
