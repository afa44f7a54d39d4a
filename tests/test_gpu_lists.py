"""The settling calls' lists of rows to re-evaluate and their maximum: many
segments (past what one scatter scans itself) of sizes around the 64-row words
and the waves' list room, with invalid rows, accept exactly what the FP64
likelihood and rejection step do; a segment with an invalid row has a NaN
maximum there and here."""
import numpy as np
import pytest
import torch

from thejoker_amd import batch as B
from thejoker_amd import device as D

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 127, 447, 448, 449, 512, 513, 4095, 4096, 4097, 20001]


def _star(N, seed, K):
    g = np.random.default_rng(seed)
    t = np.sort(g.uniform(0, 500.0, N))
    rv = K * np.sin(2 * np.pi * t / 37.0) + g.normal(0, 0.3, N) + 5.0
    return D.DeviceStar(t, rv, np.full(N, 1 / 0.09), np.ones((N, 1)), np.zeros(2),
                        np.array([900.0, 1e4]), t[0])


@pytest.mark.parametrize("n_seg", [1, 15, 64, 65, 130])
@pytest.mark.parametrize("nan_rows", [False, True])
def test_settled_rejection_equals_fp64(gpu, n_seg, nan_rows):
    stars = [_star(4 + k % 13, k, 0.0 if k % 2 else 8.0) for k in range(n_seg)]
    sizes = np.array([SIZES[k % len(SIZES)] for k in range(n_seg)])
    g = np.random.default_rng(n_seg)
    n = max(int(sizes.max()), 200)
    P = np.exp(g.uniform(np.log(2), np.log(500), n))
    if nan_rows:
        P[100] = 0.0                       # invalid in every segment past 100 rows
    cache = D.PriorCache(P, g.beta(0.867, 3.03, n), g.uniform(0, 6.28, n), g.uniform(0, 6.28, n),
                         np.exp(g.normal(-3, 1, n)))
    table = B.StarBatch(stars)
    items, off, total = B.work_items(sizes, 1024)
    d_items = B.upload_items(items)
    states = [D.pcg64_state(np.random.default_rng(1000 + k)) for k in range(n_seg)]
    ll = B.lnl_batch(table, cache, d_items, len(items), total, "f64")
    want, npw, mxw = B.reject_batch(ll, off, sizes, states, 100000)
    for call in ("settle_reject", "settle"):
        bound = torch.empty(total, dtype=torch.float32, device="cuda")
        lm = B.lnl_batch(table, cache, d_items, len(items), total, "mixed", bound=bound)
        if call == "settle_reject":
            got, npg, mxg, cnt = B.settle_reject_batch(table, cache, lm, bound, off, sizes, states,
                                                       100000)
        else:
            cnt = B.settle_batch(table, cache, lm, bound, off, sizes, states).cpu().numpy()
            got, npg, mxg = B.reject_batch(lm, off, sizes, states, 100000)
        for k in range(n_seg):
            assert np.array_equal(got[k], want[k]), (call, k)
        assert np.array_equal(npg, npw) and np.array_equal(mxg, mxw, equal_nan=True)
        b = bound.cpu().numpy()
        done = np.array([(b[o:o + m] == 0).sum() for o, m in zip(off, sizes)])
        assert np.array_equal(done, cnt)
        z = b == 0
        assert np.array_equal(lm.cpu().numpy()[z], ll.cpu().numpy()[z], equal_nan=True)
    if nan_rows:
        assert np.isnan(mxw[sizes > 100]).all() and np.isfinite(mxw[sizes <= 100]).all()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 262145, (3 << 19) - 1, 3 << 19,
                               (3 << 19) + 1])
@pytest.mark.parametrize("kind", ["peaked", "flat", "nan"])
def test_reject_dispatch_edges(gpu, n, kind):
    """Both forms of the rejection flags around the row count where they meet,
    against numpy, through the call that reduces the maximum and the one that
    is given it."""
    g = np.random.default_rng(n)
    ll = -(g.random(n) * (1e5 if kind == "peaked" else 3.0))
    if kind == "nan":
        ll[n // 2] = np.nan
    rng = np.random.default_rng(5)
    state = D.pcg64_state(rng)
    u = rng.uniform(size=n)
    with np.errstate(invalid="ignore"):
        want = np.where(np.exp(ll - ll.max()) > u)[0]
    d = torch.as_tensor(ll, device="cuda")
    idx, n_pass, mx = D.reject(d, state, n)
    assert n_pass == len(want) and np.array_equal(idx, want)
    assert np.array_equal(mx, ll.max(), equal_nan=True)
    top = torch.as_tensor([ll.max()], dtype=torch.float64, device="cuda")
    idx, n_pass, _ = D.reject(d, state, 100, llmax=top)
    assert n_pass == len(want) and np.array_equal(idx, want[:100])


@pytest.mark.parametrize("n_seg", [1, 4, 5])
def test_descriptor_upload_edges(gpu, n_seg):
    """Descriptors as kernel arguments (up to four segments) and by a copy:
    two calls queued one after the other, each on other segments, give what
    they give alone, segment by segment."""
    g = np.random.default_rng(n_seg)
    sizes = [700 + 131 * i for i in range(n_seg)]
    off = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    ll = torch.as_tensor(g.normal(-20.0, 3.0, int(sum(sizes))), device="cuda")
    ll2 = torch.as_tensor(g.normal(-5.0, 1.0, int(sum(sizes))), device="cuda")
    states = [(int(g.integers(1 << 62)) << 60 | 5, int(g.integers(1 << 62)) | 1)
              for _ in range(n_seg)]
    for x in (ll, ll2):
        idx, n_pass, mx = B.reject_batch(x, off, sizes, states, 50)
        for i in range(n_seg):
            one = B.reject_batch(x[off[i]:off[i] + sizes[i]].clone(), [0], [sizes[i]],
                                 [states[i]], 50)
            assert np.array_equal(idx[i], one[0][0]) and n_pass[i] == one[1][0]
            assert mx[i] == one[2][0] == float(x[off[i]:off[i] + sizes[i]].max())


def test_segment_maximum_edges(gpu):
    """Segments whose maximum comes from one partial, from several, and from
    more than a workgroup has threads, one with a NaN, side by side, against
    numpy."""
    g = np.random.default_rng(11)
    sizes = [1, 4096, 4097, 300 * 4096 + 5, 64, 10000]
    off = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    ll = -(g.random(int(sum(sizes))) * 5.0)
    ll[off[5] + 9999] = np.nan
    ll[off[3] + sizes[3] - 1] = 1.0          # the last row of the last partial
    states, us = [], []
    for i, n in enumerate(sizes):
        rng = np.random.default_rng(100 + i)
        states.append(D.pcg64_state(rng))
        us.append(rng.uniform(size=n))
    idx, n_pass, mx = B.reject_batch(torch.as_tensor(ll, device="cuda"), off, sizes, states, 500)
    for i, n in enumerate(sizes):
        x = ll[off[i]:off[i] + n]
        want = np.where(np.exp(x - x.max()) > us[i])[0]
        assert n_pass[i] == len(want) and np.array_equal(idx[i], want[:500])
        assert np.array_equal(mx[i], x.max(), equal_nan=True)
