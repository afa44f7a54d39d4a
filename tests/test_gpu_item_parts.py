"""Work items split into parts of whole workgroup passes: item sizes around a
workgroup, item counts and explicit grids that give one, two, four and eight
parts, against the single-star launch bit for bit; the pruned launch the same
with its probe off (every row evaluated and counted once)."""
import numpy as np
import pytest
import torch

from thejoker_amd import batch as B
from thejoker_amd import device as D
from thejoker_amd import synthetic as syn

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 255, 256, 257, 511, 1025, 2047, 2048]


@pytest.fixture(scope="module")
def setup(gpu):
    cols = syn.prior_columns(1 << 12, seed=19, jitter=True)
    cache = D.PriorCache(cols["P"], cols["e"], cols["omega"], cols["M0"], cols["s"])
    devs = []
    for st in syn.many_stars(len(SIZES), seed=8):
        devs.append(D.DeviceStar(st.t, st.rv, st.ivar(), st.trend(), np.zeros(2),
                                 np.array([900.0, 1e4]), st.t_ref, jitter_mode="physical"))
    return devs, cache


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("block,grid", [(256, 0), (256, 1), (256, 12), (256, 23), (128, 6),
                                        (64, 0), (64, 44)])
def test_parts_equal_single(setup, precision, block, grid):
    devs, cache = setup
    table = B.StarBatch(devs)
    shape = B.LaunchShape(block, grid, 2048)
    begin = [17 * i for i in range(len(SIZES))]
    items, off, total = B.work_items(SIZES, shape.tile, row_begin=begin)
    d_items = B.upload_items(items)
    mixed = precision == "mixed"
    out = torch.full((total + 64,), 5.0, dtype=torch.float64, device="cuda")
    bnd = torch.full((total + 64,), 5.0, dtype=torch.float32, device="cuda") if mixed else None
    B.lnl_batch(table, cache, d_items, len(items), total, precision, shape, out=out, bound=bnd)
    got = out.cpu().numpy()
    assert (got[total:] == 5.0).all()
    prune = torch.as_tensor(np.tile([-np.inf, 0.0], len(SIZES)), device="cuda")
    out2 = torch.full((total + 64,), 5.0, dtype=torch.float64, device="cuda")
    bnd2 = torch.full((total + 64,), 5.0, dtype=torch.float32, device="cuda")
    n_full = torch.zeros(len(SIZES), dtype=torch.int64, device="cuda")
    B.lnl_prune_batch(table, table, prune, cache, d_items, len(items), precision, shape, out=out2,
                      bound=bnd2, n_full=n_full)
    assert np.array_equal(out2.cpu().numpy(), got, equal_nan=True)
    assert n_full.cpu().tolist() == SIZES
    for i, (d, n) in enumerate(zip(devs, SIZES)):
        sl = slice(off[i], off[i] + n)
        want = D.lnl(d, cache, precision=precision).cpu().numpy()[begin[i]:begin[i] + n]
        assert np.array_equal(got[sl], want, equal_nan=True), i
        if mixed:
            assert np.array_equal(bnd.cpu().numpy()[sl], bnd2.cpu().numpy()[sl], equal_nan=True)
