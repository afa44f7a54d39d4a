"""`grid` of a many-star launch caps its workgroups: the same values whatever the
cap, one workgroup included, for whole items and parts, empty items among them,
plain and pruned; and a launch of two workgroups takes many times as long as one
that fills the device, as it leaves the rest of it to other streams."""
import numpy as np
import pytest
import torch

from thejoker_amd import batch as B
from thejoker_amd import device as D
from thejoker_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(gpu):
    cols = syn.prior_columns(1 << 13, seed=19, jitter=True)
    cache = D.PriorCache(cols["P"], cols["e"], cols["omega"], cols["M0"], cols["s"])
    devs = [D.DeviceStar(st.t, st.rv, st.ivar(), st.trend(), np.zeros(2), np.array([900.0, 1e4]),
                         st.t_ref, jitter_mode="physical") for st in syn.many_stars(7, seed=8)]
    return devs, B.StarBatch(devs), cache


def _launch(setup, precision, prune, shape, items, total):
    devs, table, cache = setup
    out = torch.full((total,), 5.0, dtype=torch.float64, device="cuda")
    bnd = torch.full((total,), 5.0, dtype=torch.float32, device="cuda")
    d_items = B.upload_items(items)
    if not prune:
        B.lnl_batch(table, cache, d_items, len(items), total, precision, shape, out=out,
                    bound=bnd if precision == "mixed" else None)
        return out.cpu().numpy(), bnd.cpu().numpy(), None
    n_full = torch.zeros(len(table), dtype=torch.int64, device="cuda")
    # every second star probed (by itself: its own value is a bound), half of them pruned
    thr = np.where(np.arange(7) % 2, -np.inf, np.where(np.arange(7) % 4, np.inf, -50.0))
    d_prune = torch.as_tensor(np.stack([thr, np.zeros(7)], 1).reshape(-1), device="cuda")
    B.lnl_prune_batch(table, table, d_prune, cache, d_items, len(items), precision, shape, out=out,
                      bound=bnd, n_full=n_full)
    return out.cpu().numpy(), bnd.cpu().numpy(), n_full.cpu().numpy()


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("prune", [False, True])
def test_same_values_under_any_cap(setup, precision, prune):
    sizes = [1, 300, 2048, 2049, 5000, 64, 8000]
    items, off, total = B.work_items(sizes, 700)
    empty = items[:1].copy()
    empty["n_rows"] = 0
    items = np.concatenate([items[:3], empty, items[3:]])
    want = _launch(setup, precision, prune, B.LaunchShape(256, 0, 700), items, total)
    for block, grid in [(256, 1), (256, 3), (128, 7), (64, 200), (256, 100000)]:
        got = _launch(setup, precision, prune, B.LaunchShape(block, grid, 700), items, total)
        for a, b in zip(got, want):
            assert (a is None) == (b is None) and (a is None or np.array_equal(a, b,
                                                                              equal_nan=True))


def test_cap_holds(setup):
    devs, table, cache = setup
    items, off, total = B.work_items([8192] * 7, 512)
    items = np.concatenate([items] * 8)
    d_items = B.upload_items(items)
    out = torch.empty(total, dtype=torch.float64, device="cuda")

    def ms(grid):
        shape = B.LaunchShape(256, grid, 512)
        B.lnl_batch(table, cache, d_items, len(items), total, "f64", shape, out=out)
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(3):
            B.lnl_batch(table, cache, d_items, len(items), total, "f64", shape, out=out)
        b.record()
        b.synchronize()
        return a.elapsed_time(b)

    assert ms(2) > 5 * ms(0)
