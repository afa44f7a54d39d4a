"""Segmented calls behind work still running on the stream: those documented to
synchronise it return with it idle, for one segment as for many (a caller may
read their results through another stream); the others leave it running, and two
of them queued one behind the other, with different descriptors over the same
scratch, give what each gives by itself."""
import ctypes

import numpy as np
import pytest
import torch

from thejoker_amd import _lib
from thejoker_amd import batch as B
from thejoker_amd import device as D

pytestmark = pytest.mark.gpu

ROWS = 3000


class Setup:
    def __init__(self):
        g = np.random.default_rng(3)
        n = 1 << 21
        self.cache = D.PriorCache(np.exp(g.uniform(1, 6, n)), g.beta(0.867, 3.03, n),
                                  g.uniform(0, 6.28, n), g.uniform(0, 6.28, n),
                                  np.exp(g.normal(-3, 1, n)))
        self.stars = [self.star(8 + k, k) for k in range(6)]
        self.long_star = self.star(200, 99)
        self.table = B.StarBatch(self.stars)
        self.states = [D.pcg64_state(np.random.default_rng(k)) for k in range(6)]
        self.out = torch.empty(n, dtype=torch.float64, device="cuda")

    @staticmethod
    def star(N, seed):
        g = np.random.default_rng(seed)
        t = np.sort(g.uniform(0, 500.0, N))
        return D.DeviceStar(t, g.normal(0, 3, N), np.full(N, 1 / 0.09), np.ones((N, 1)),
                            np.zeros(2), np.array([900.0, 1e4]), t[0])

    def busy(self):
        """A few milliseconds of work on the stream."""
        for _ in range(4):
            D.lnl(self.long_star, self.cache, out=self.out)

    def mixed(self, n_seg):
        sizes = np.full(n_seg, ROWS)
        items, off, total = B.work_items(sizes, 1024)
        bound = torch.empty(total, dtype=torch.float32, device="cuda")
        ll = B.lnl_batch(self.table, self.cache, B.upload_items(items), len(items), total, "mixed",
                         bound=bound)
        torch.cuda.synchronize()
        return ll, bound, off, sizes


@pytest.fixture(scope="module")
def setup(gpu):
    return Setup()


def _idle():
    return torch.cuda.current_stream().query()


@pytest.mark.parametrize("n_seg", [1, 4, 5])
@pytest.mark.parametrize("call", ["settle", "live", "polish", "reject", "zero_check",
                                  "settle_reject"])
def test_documented_waits(setup, call, n_seg):
    ll, bound, off, sizes = setup.mixed(n_seg)
    lib = _lib.ensure_device(0)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    vp = lambda x: ctypes.c_void_p(x.data_ptr())
    res = torch.zeros((4, n_seg), dtype=torch.int64, device="cuda")
    idx = torch.zeros(n_seg * 50, dtype=torch.int64, device="cuda")
    c = setup.cache
    cols = [vp(x) for x in (c.P, c.e, c.omega, c.M0, c.s)]
    setup.busy()
    assert not _idle()
    if call == "settle":
        B.settle_batch(setup.table, c, ll, bound, off, sizes, setup.states[:n_seg])
    elif call == "live":
        B.settle_live_batch(setup.table, c, ll, bound, off, sizes, [0] * n_seg, [-np.inf] * n_seg)
    elif call == "polish":
        B.polish_batch(setup.table, c, ll, off, sizes)
    elif call == "settle_reject":
        segs = np.zeros(n_seg, dtype=B.SETTLE_SEGMENT_DTYPE)
        segs["offset"], segs["n"], segs["star"] = off, sizes, np.arange(n_seg)
        _lib.check(lib.jk_settle_reject_batch(
            setup.table.handle, n_seg, segs.ctypes.data_as(ctypes.c_void_p), 50, *cols,
            ctypes.c_void_p(0), vp(ll), vp(bound), vp(idx), vp(res[0]), vp(res[1]), vp(res[2]), st))
    else:
        segs = np.zeros(n_seg, dtype=B.SEGMENT_DTYPE)
        segs["offset"], segs["n"], segs["max_keep"] = off, sizes, 50
        segs["idx_offset"] = 50 * np.arange(n_seg)
        args = [vp(ll), n_seg, segs.ctypes.data_as(ctypes.c_void_p), vp(idx), vp(res[0]),
                vp(res[1])]
        if call == "reject":
            _lib.check(lib.jk_reject_batch(*args, st))
        else:
            _lib.check(lib.jk_reject_batch_zero_check(*args, vp(res[2]), st))
    assert _idle()


@pytest.mark.parametrize("n_a,n_b", [(1, 4), (4, 1), (3, 2), (2, 5)])
@pytest.mark.parametrize("call", ["tol", "pruned"])
def test_queued_behind_one_another(setup, call, n_a, n_b):
    def run(work, n_seg, stars):
        ll, bound, off, sizes = work
        if call == "tol":
            return B.settle_tol_batch(setup.table, setup.cache, ll, bound, off, sizes, stars=stars,
                                      tol=1e-5)
        return B.settle_pruned_batch(setup.table, setup.cache, ll, bound, off, sizes, stars=stars)

    def inputs(n_seg):
        ll, bound, off, sizes = setup.mixed(n_seg)
        if call == "pruned":
            bound[::2] = -1.0           # upper bounds
            torch.cuda.synchronize()
        return ll, bound, off, sizes

    stars = {n: np.arange(n)[::-1].copy() for n in (n_a, n_b)}
    alone = []
    for n in (n_a, n_b):
        w = inputs(n)
        alone.append((run(w, n, stars[n]).cpu().numpy(), w[0].cpu().numpy(), w[1].cpu().numpy()))
    wa, wb = inputs(n_a), inputs(n_b)
    setup.busy()
    cnt_a = run(wa, n_a, stars[n_a])
    if n_a <= 4:
        assert not _idle()
    cnt_b = run(wb, n_b, stars[n_b])
    for (cnt, ll, bound), c, w in zip(alone, (cnt_a, cnt_b), (wa, wb)):
        assert np.array_equal(c.cpu().numpy(), cnt) and int(cnt.sum()) > 0
        assert np.array_equal(w[0].cpu().numpy(), ll, equal_nan=True)
        assert np.array_equal(w[1].cpu().numpy(), bound)
