"""The raw search op on rows and tables that no grid of this package gives: rows outside the grid or of another bin, and
boundary tables that end early. Nothing is read beyond a table, and what the table holds is answered."""
import numpy as np
import pytest
import torch

from test_data_errors import _status_after
from test_gpu_collected_search import brute_force

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SPLITS = [0, 250, 600]


class Binned:
    """two events in bin order with the tables of the reference's own binning, and the op on them"""

    def __init__(self, oracle, dims, n_bins=5):
        rng = np.random.default_rng(dims)
        x = rng.random((SPLITS[-1], dims)).astype(np.float32)
        self.rows, self.flat, self.n_bins, self.width, count = oracle.BinByCoordinates(x, np.array(SPLITS, np.int32), n_bins=n_bins)
        order = np.argsort(self.flat, kind="stable")
        self.x, self.rows, self.flat = x[order], self.rows[order].copy(), self.flat[order]
        self.bounds = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
        self.cells = int(np.prod(self.n_bins))

    def search(self, K, radius=0.0, table=None, rows=None):
        """indices, squared distances and the flags that the call left"""
        from hgcalml_amd._lib import check, lib, p, stream
        on_gpu = [torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
                  for a in (self.x, self.flat, self.rows if rows is None else rows, self.bounds if table is None else table,
                            self.n_bins, self.width)]
        x, flat, rows, table, n_bins, width = on_gpu
        n, dims = x.shape
        idx = torch.empty((n, K), dtype=torch.int32, device=DEV)
        dist = torch.empty((n, K), dtype=torch.float32, device=DEV)
        flags = _status_after(lambda: check(lib.hgc_binned_select_knn_fused(
            p(x), p(flat), None, p(rows), p(table), p(n_bins), p(width), None, None, radius or -1.0, p(idx), p(dist), n, K, dims,
            dims, len(table), 0, 0, stream())))
        return idx.cpu(), dist.cpu(), flags


def wrong_rows(binned, kind):
    """every seventh row names a bin outside the grid, or one of the grid that is not the point's own"""
    rows = binned.rows.copy()
    some = np.arange(0, len(rows), 7)
    rng = np.random.default_rng(1)
    if kind == "above":
        rows[some, -1] = binned.n_bins[-1] + rng.integers(0, 40, len(some))
    elif kind == "far above":
        rows[some, -1] = 1 << 20
    elif kind == "event":  # the entry that names the event is not looked at
        rows[some, 0] = rng.integers(-2, 3, len(some))
    elif kind == "below":
        rows[some, 1] = -1 - rng.integers(0, 40, len(some))
    else:
        rows[some, 1:] = rng.integers(0, binned.n_bins, (len(some), len(binned.n_bins)))
    return rows


@pytest.mark.parametrize("dims", [2, 3, 4, 5])
@pytest.mark.parametrize("kind", ["above", "far above", "below", "another", "event"])
@pytest.mark.parametrize("K,radius", [(6, 0.0), (6, 0.2), (100, 0.0), (140, 0.0), (140, 0.2)])
def test_rows_that_do_not_name_the_own_bin(oracle, dims, kind, K, radius):
    """such a row says nothing about where its point is: the whole event is searched, of the event that its bin names"""
    from hgcalml_amd import ops
    binned = Binned(oracle, dims)
    want = brute_force(torch.from_numpy(binned.x), SPLITS, K, radius, None)
    idx, dist, flags = binned.search(K, radius, rows=wrong_rows(binned, kind))
    assert flags == 0
    assert torch.equal(idx, want[0]) and torch.equal(dist, want[1])
    # the table ends with the first event: the second one's points have no neighbours
    idx, dist, flags = binned.search(K, radius, table=binned.bounds[:binned.cells + 1], rows=wrong_rows(binned, kind))
    assert flags == ops.FLAG_BIN_BEYOND_TABLE
    first = SPLITS[1]
    assert torch.equal(idx[:first], want[0][:first]) and torch.equal(dist[:first], want[1][:first])
    assert (idx[first:, 1:] == -1).all() and (dist[first:] == 0).all()


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K", [6, 140])  # collected, and by shells
@pytest.mark.parametrize("n_bins", [3, 4, 5])
@pytest.mark.parametrize("where", ["below", "the largest integer"])
def test_bins_outside_every_event_have_no_neighbours(oracle, dims, K, n_bins, where):
    from hgcalml_amd import ops
    binned = Binned(oracle, dims, n_bins)
    want = binned.search(K)
    bad = torch.arange(len(binned.x)) % 11 == 0
    binned.flat[bad.numpy()] = -binned.cells - 3 if where == "below" else (1 << 31) - 1
    idx, dist, flags = binned.search(K)
    assert want[2] == 0 and flags == ops.FLAG_BIN_BEYOND_TABLE
    assert torch.equal(idx[~bad], want[0][~bad]) and torch.equal(dist[~bad], want[1][~bad])
    assert (idx[bad, 1:] == -1).all() and (dist[bad] == 0).all()


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K,radius", [(6, 0.0), (6, 0.2), (140, 0.0)])  # collected, and by shells
@pytest.mark.parametrize("share", [0.1, 0.5, 0.93])
def test_table_that_ends_inside_an_event(oracle, dims, K, radius, share):
    """bins beyond the table hold nothing, the bins in front of its end keep their points (the rows of a point whose own
    bin is beyond the table are left open)"""
    from hgcalml_amd import ops
    binned = Binned(oracle, dims)
    n_bins_left = binned.cells + int(share * binned.cells)
    x = torch.from_numpy(binned.x)
    left = int(binned.bounds[n_bins_left])  # points in bin order
    want = brute_force(x[:left], [0, SPLITS[1], left], K, radius, None)
    idx, dist, flags = binned.search(K, radius, table=binned.bounds[:n_bins_left + 1])
    assert flags == ops.FLAG_BIN_BEYOND_TABLE
    assert torch.equal(idx[:left], want[0]) and torch.equal(dist[:left], want[1])
    assert (idx[left:] < left).logical_or(idx[left:] == torch.arange(left, len(idx))[:, None]).all()


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K", [6, 140])
@pytest.mark.parametrize("at,value", [(0, 0), (-1, 0), (0, -7), (-1, -7), (-1, 1 << 30)])
def test_numbers_of_bins_that_no_grid_has(oracle, dims, K, at, value):
    """the call ends, reports it and reads nothing beyond the table"""
    from hgcalml_amd import ops
    binned = Binned(oracle, dims)
    binned.n_bins = binned.n_bins.copy()
    binned.n_bins[at] = value
    idx, dist, flags = binned.search(K)
    assert flags == ops.FLAG_BIN_BEYOND_TABLE
    assert (idx[:, 0] == torch.arange(len(idx))).all() and (idx[:, 1:] < len(idx)).all()


@pytest.mark.parametrize("dims,n_bins,events", [(3, 102, 16), (2, 2100, 4), (4, 64, 2)])
@pytest.mark.parametrize("K", [9, 140])
def test_tables_of_2_to_the_24_bins_and_more(dims, n_bins, events, K):
    """bins per dimension are few, the bins of all events many: the same answers"""
    from hgcalml_amd import ops
    from hgcalml_amd._lib import check, lib, p, stream
    gen = torch.Generator().manual_seed(dims)
    n = 150 * events + 7
    x = torch.rand(n, dims, generator=gen)
    splits = [150 * e for e in range(events)] + [n]
    bins = torch.tensor([n_bins] * dims, dtype=torch.int32, device=DEV)
    width = torch.tensor([1.0 / n_bins], device=DEV)
    total = events * n_bins ** dims
    assert total >= 1 << 24
    on_gpu = x.to(DEV)
    rows, flat, count = torch.ops.hgcalml.bin_by_coordinates(on_gpu, torch.tensor(splits, dtype=torch.int32, device=DEV), width,
                                                             bins, total, True)
    order = torch.argsort(flat.long() * n + torch.arange(n, device=DEV))
    table = torch.zeros(total + 1, dtype=torch.int32, device=DEV)
    table[1:] = torch.cumsum(count, 0, dtype=torch.int32)
    idx = torch.empty((n, K), dtype=torch.int32, device=DEV)
    dist = torch.empty((n, K), dtype=torch.float32, device=DEV)
    a = [on_gpu[order].contiguous(), flat[order].contiguous(), rows[order].contiguous()]
    sorting = order.to(torch.int32)
    flags = _status_after(lambda: check(lib.hgc_binned_select_knn_fused(
        p(a[0]), p(a[1]), None, p(a[2]), p(table), p(bins), p(width), p(sorting), None, -1.0, p(idx), p(dist), n, K, dims, dims,
        len(table), 0, 0, stream())))
    want = brute_force(x, splits, K, 0.0, None)
    assert flags in (0, ops.FLAG_COORDINATE_OUT_OF_GRID)
    assert torch.equal(idx.cpu(), want[0]) and torch.equal(dist.cpu(), want[1])


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K", [5, 17, 65, 129, 140])
@pytest.mark.parametrize("again", [0, 1, 5, 650])
def test_a_sorting_that_names_one_point_many_times(oracle, dims, K, again):
    """300 points in one place are all called `again`: equal keys, more than the buffer of the collected search holds"""
    from hgcalml_amd._lib import check, lib, p, stream
    rng = np.random.default_rng(dims)
    n = 1000
    x = rng.random((n, dims)).astype(np.float32)
    x[200:800] = 0.5
    names = rng.permutation(n).astype(np.int32)
    names[450:750] = again  # all of them in that place
    rows, flat, n_bins, width, count = oracle.BinByCoordinates(x, np.array([0, n], np.int32), n_bins=4)
    order = np.argsort(flat, kind="stable")
    x, rows, flat, names = x[order], rows[order], flat[order], names[order]
    bounds = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    on_gpu = [torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in (x, flat, rows, bounds, n_bins, width, names)]
    gx, gflat, grows, gbounds, gbins, gwidth, gnames = on_gpu
    idx = torch.zeros((n, K), dtype=torch.int32, device=DEV)
    dist = torch.zeros((n, K), dtype=torch.float32, device=DEV)
    check(lib.hgc_binned_select_knn_fused(p(gx), p(gflat), None, p(grows), p(gbounds), p(gbins), p(gwidth), p(gnames), None, -1.0,
                                          p(idx), p(dist), n, K, dims, dims, len(bounds), 0, 0, stream()))
    idx, dist = idx.cpu().numpy(), dist.cpu().numpy()
    d = np.zeros((n, n), np.float32)
    for c in range(dims):
        step = x[:, None, c] - x[None, :, c]
        d = d + step * step
    key = (d.view(np.uint32).astype(np.uint64) << np.uint64(32)) | names.astype(np.uint64)[None, :]
    np.fill_diagonal(key, np.iinfo(np.uint64).max)
    key = np.sort(key, axis=1)[:, :K - 1]
    once = np.flatnonzero(np.bincount(names, minlength=n)[names] == 1)  # the rows that one point writes
    assert (idx[names[once], 1:] == (key[once] & np.uint64(0xffffffff)).astype(np.int32)).all()
    assert (dist[names[once], 1:].view(np.uint32) == (key[once] >> np.uint64(32)).astype(np.uint32)).all()


@pytest.mark.parametrize("dims", [2, 3, 4])
@pytest.mark.parametrize("K", [6, 140])
def test_the_largest_integer_as_a_bin_of_a_grid_that_divides_it(oracle, dims, K):
    """its event would end exactly where the integers do; the other rows are those of another grid and left open"""
    from hgcalml_amd import ops
    binned = Binned(oracle, dims)
    binned.n_bins = np.full(dims, 4, np.int32)
    bad = torch.arange(len(binned.x)) % 11 == 0
    binned.flat[bad.numpy()] = (1 << 31) - 1
    idx, dist, flags = binned.search(K)
    assert flags & ops.FLAG_BIN_BEYOND_TABLE
    assert (idx[bad, 1:] == -1).all() and (dist[bad] == 0).all()
