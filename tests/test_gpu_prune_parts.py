"""Pruned launches over item counts around the lines at which an item is one,
two and four parts, over the numbers of linear parameters: a row that is not
pruned gets exactly the unpruned launch's value (and bound), a pruned one a
value below the threshold and not below its lnL, and each is counted once."""
import numpy as np
import pytest
import torch

from thejoker_amd import batch as B
from thejoker_amd import device as D
from thejoker_amd import synthetic as syn

pytestmark = pytest.mark.gpu

TILE = 128


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("jitter", [True, False])
@pytest.mark.parametrize("poly,offsets", [(1, 0), (1, 2), (2, 2), (3, 2)])
def test_pruned_rows(gpu, poly, offsets, jitter, precision):
    st = syn.many_stars(1, seed=4, M_range=(40, 41))[0]
    trend = st.trend(poly_trend=poly)
    groups = np.arange(st.M) % (offsets + 1)
    trend = np.concatenate([trend] + [(groups == g)[:, None] for g in range(1, offsets + 1)], 1)
    L = 1 + trend.shape[1]
    lam = np.array([900.0, 1e4, 0.25, 1e-6][:1 + poly] + [25.0] * offsets)
    a = dict(t=st.t, rv=st.rv, ivar=st.ivar(), trend=trend, mu=np.zeros(L), lam=lam,
             t_ref=st.t_ref, cov=None, k_prior_mode=0, sigma_K0=30.0, P0=365.25, max_K=300.0)
    mode = "physical" if jitter else "reference"
    star = D.DeviceStar(a["t"], a["rv"], a["ivar"], a["trend"], a["mu"], a["lam"], a["t_ref"],
                        jitter_mode=mode)
    probe, add = D.probe_star(a, mode)
    n_max = 513 * TILE - 63
    cols = syn.prior_columns(n_max, seed=6, jitter=True)
    cache = D.PriorCache(cols["P"], cols["e"], cols["omega"], cols["M0"], cols["s"])
    ref = D.lnl(star, cache).cpu().numpy()
    thr = np.nanmedian(D.lnl(probe, cache).cpu().numpy()) + add    # about half are pruned
    table, probes = B.StarBatch([star]), B.StarBatch([probe])
    prune = torch.as_tensor([thr, add], dtype=torch.float64, device="cuda")
    mixed = precision == "mixed"
    n_cut = 0
    for k in (1, 128, 129, 256, 257, 513):
        n = k * TILE - (63 if k > 1 else 0)
        shape = B.LaunchShape(64, 0, TILE)
        items, off, total = B.work_items([n], TILE)
        assert len(items) == k and total == n
        d_items = B.upload_items(items)
        b0 = torch.empty(total, dtype=torch.float32, device="cuda") if mixed else None
        want = B.lnl_batch(table, cache, d_items, k, total, precision, shape,
                           bound=b0).cpu().numpy()
        b1 = torch.full((total,), 7.0, dtype=torch.float32, device="cuda")
        out = torch.full((total,), 7.0, dtype=torch.float64, device="cuda")
        n_full = torch.zeros(1, dtype=torch.int64, device="cuda")
        B.lnl_prune_batch(table, probes, prune, cache, d_items, k, precision, shape, out=out,
                          bound=b1, n_full=n_full)
        got, bound = out.cpu().numpy(), b1.cpu().numpy()
        cut = bound == -1.0
        assert cut.sum() + int(n_full[0]) == n, k
        n_cut += int(cut.sum())
        assert np.array_equal(got[~cut], want[~cut], equal_nan=True), k
        assert (got[cut] < thr).all() and (got[cut] >= ref[:n][cut]).all(), k
        if mixed:
            assert np.array_equal(bound[~cut], b0.cpu().numpy()[~cut]), k
    assert n_cut > 0
